"""Steps of few single tokens through all layers in one launch (``csrc/chain.hip``, ``chain_f32.hip``), or of one short prompt
(``chain_prompt.hip``), against the layers' own kernels: single tokens in bfloat16 the same bits in groups of up to
four heads, else both measured by the 32-bit path on the same weights; in 32 bits both measured by the oracle in 64.  Sizes are
those at which the launch changes what it does: a K that leaves waves without a chunk or takes them a second round, groups of heads
beyond four, four and eight waves, runs of the keys."""

import numpy as np
import pytest
import torch

from configs import llama
from nnis_amd.errors import KernelError, StepLost

pytestmark = pytest.mark.gpu


def _config(width, heads, kv_heads, inner, layers=2):
    return llama(num_hidden_layers=layers, hidden_size=width, num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=64,
                 intermediate_size=inner, vocab_size=509, rope_theta=10000.0, rms_norm_eps=1e-5, tie_word_embeddings=True,
                 max_position_embeddings=4096, torch_dtype="bfloat16")


# width, query heads, key heads, inner size
SIZES = [
    (64, 1, 1, 64),        # one chunk of K: three of four waves have no share of it
    (320, 5, 1, 128),      # a group of five heads
    (192, 6, 2, 1600),     # down takes 25 chunks: a wave's second round of weights
    (1024, 14, 7, 448),    # the widest of four waves
    (576, 9, 3, 1536),     # the 135M shape's
    (1088, 8, 8, 576),     # eight waves, 17 chunks; a head a key head
    (1152, 16, 4, 5184),   # down takes 81 chunks, the even and the odd apart; gate and up in 4 parts
    (1152, 16, 2, 8256),   # down takes 129 chunks
]
# lengths before the step: the first token, pages' ends, runs
LENGTHS = [1, 63, 64, 65, 200, 1023, 1100, 5, 128, 320, 577, 129, 31, 2000, 90, 447]


def _tokens(lengths, steps):
    rng = np.random.default_rng(sum(lengths))
    return [rng.integers(0, 509, size=n).tolist() for n in lengths], [rng.integers(0, 509, size=len(lengths)).tolist() for _ in range(steps)]


def _run(folder, dtype, lengths, plan, monkeypatch, steps=3):
    """The logits of ``steps`` steps of single tokens behind prompts of these lengths, [steps, sequences, vocab]."""
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry
    from nnis_amd.kernels import ops

    with monkeypatch.context() as patch:
        patch.setattr(ops, "chain_prompt_takes", lambda *args, **sizes: False)  # (the same cache for all)
        if plan != "own":
            patch.setattr(ops, "chain_plan", lambda *args, **sizes: plan)
        engine = load_engine(folder, dtype=dtype, max_tokens=sum(-(-(n + steps + 1) // 64) * 64 for n in lengths))
        prompts, tokens = _tokens(lengths, steps)
        slots = [engine.start_sequence() for _ in lengths]
        engine.step([StepEntry(slot, prompt, None) for slot, prompt in zip(slots, prompts)])
        out = []
        for step in range(steps):
            entries = [StepEntry(slot, [token], None) for slot, token in zip(slots, tokens[step])]
            out.append(engine.step(entries).double().cpu())
            if len(out) == 1:  # the same step again, replayed over what the first left in the exchange
                for slot, n in zip(slots, lengths):
                    engine.truncate(slot, n)
                assert torch.equal(engine.step(entries).double().cpu(), out[0])
        chain = engine.model.layer_chain(engine.rt)
        ran = chain is not None and len(chain.tables) > 0
        return torch.stack(out), ran, engine


@pytest.mark.parametrize("sizes", [(64, 1, 1, 64), (192, 6, 2, 1600), (576, 9, 3, 1536), (1024, 14, 7, 448), (1024, 16, 16, 2048)])
def test_two_tiles_of_rows(tmp_path, sizes, monkeypatch):
    """17 to 32 rows of narrow models: the layers' bits."""
    import nnis_amd

    nnis_amd.write_random_model(str(tmp_path), _config(*sizes), 3)
    for batch in (17, 20, 32):
        lengths = (LENGTHS + [n + 1 for n in LENGTHS])[:batch]
        layers, ran, _ = _run(str(tmp_path), "bfloat16", lengths, None, monkeypatch)
        assert not ran
        got, ran, _ = _run(str(tmp_path), "bfloat16", lengths, "own", monkeypatch)
        assert ran and torch.equal(got, layers), batch
    assert not _run(str(tmp_path), "bfloat16", LENGTHS * 2 + [7], "own", monkeypatch)[1]


@pytest.mark.parametrize("batch", [1, 3, 16])
@pytest.mark.parametrize("sizes", SIZES)
def test_against_the_layers(tmp_path, sizes, batch, monkeypatch):
    """The same bits in groups of up to four heads, else as far from 32 bits as the layers' kernels.  (The roundings are the same;
    which of them fall together is not: over a few hundred logits the distances are within a third.)"""
    import nnis_amd

    nnis_amd.write_random_model(str(tmp_path), _config(*sizes), 3)
    lengths = LENGTHS[:batch] if batch > 1 else [1100]
    want, ran, _ = _run(str(tmp_path), "float32", lengths, None, monkeypatch)
    assert not ran
    layers, ran, _ = _run(str(tmp_path), "bfloat16", lengths, None, monkeypatch)
    assert not ran
    bound = 1.33 * (layers - want).norm()
    waves, group = 4 if sizes[0] <= 1024 else 8, sizes[1] // sizes[2]
    for plan in ("own", (1, waves), (2, waves // 2), (16, waves)):
        got, ran, _ = _run(str(tmp_path), "bfloat16", lengths, plan, monkeypatch)
        assert ran == (plan != "own" or group <= 4 or batch < 8), f"plan {plan}: whether the launch was made"
        if plan == "own" and group <= 4:
            assert torch.equal(got, layers)
        error = (got - want).norm()
        assert error <= bound, f"plan {plan}: {error.item():.4g} from 32 bits, the layers' kernels {(layers - want).norm().item():.4g}"


@pytest.mark.parametrize("batch", [5, 7, 8])
@pytest.mark.parametrize("sizes", [(320, 5, 1, 128), (1152, 16, 2, 8256)])
def test_five_to_seven_rows_of_large_groups(tmp_path, sizes, batch, monkeypatch):
    """A step's rows are padded to seven, which the launch takes, and not to eight, which it does not: as far from 32 bits as the layers'
    kernels (``test_against_the_layers``)."""
    import nnis_amd

    nnis_amd.write_random_model(str(tmp_path), _config(*sizes), 3)
    want = _run(str(tmp_path), "float32", LENGTHS[:batch], None, monkeypatch)[0]
    layers = _run(str(tmp_path), "bfloat16", LENGTHS[:batch], None, monkeypatch)[0]
    got, ran, _ = _run(str(tmp_path), "bfloat16", LENGTHS[:batch], "own", monkeypatch)
    assert ran == (batch < 8)
    assert (got - want).norm() <= 1.33 * (layers - want).norm()


@pytest.mark.parametrize("batch", [1, 3, 16])
@pytest.mark.parametrize("sizes", SIZES + [(128, 12, 1, 192)])  # (twelve heads a key head)
def test_32_bits_against_the_oracle(tmp_path, sizes, batch, monkeypatch):
    """As close to 64 bits as the layers' 32-bit kernels.  (Each sum is of the same terms in an order of its own, so the distances are
    two draws of the same size; over a few hundred logits of a few rows they are within a third.)"""
    import nnis_amd
    import plain_llama

    nnis_amd.write_random_model(str(tmp_path), dict(_config(*sizes), torch_dtype="float32"), 3)
    lengths = LENGTHS[:batch] if batch > 1 else [1100]
    prompts, tokens = _tokens(lengths, 3)
    plain = plain_llama.PlainLlama(str(tmp_path), torch.float64)
    want = torch.stack([plain.logits(prompt + [row[at] for row in tokens])[-3:] for at, prompt in enumerate(prompts)], dim=1)
    layers, ran, _ = _run(str(tmp_path), "float32", lengths, None, monkeypatch)
    assert not ran
    bound = 1.33 * (layers - want).norm()
    for plan in ("own", (1, 8), (2, 8), (16, 8)):
        got, ran, _ = _run(str(tmp_path), "float32", lengths, plan, monkeypatch)
        assert ran, f"plan {plan}: the launch was not made"
        error = (got - want).norm()
        assert error <= bound, f"plan {plan}: {error.item():.4g} from 64 bits, the layers' kernels {(layers - want).norm().item():.4g}"


def _streams(folder, lengths, plan, monkeypatch):
    """The 32-bit stream behind the last attention and what the last feed-forward adds to it, of two steps of single tokens, and whether
    the launch ran.  (Logits are of 16-bit rows, in which most differences of the last bit are gone.)"""
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry
    from nnis_amd.kernels import ops

    with monkeypatch.context() as patch:
        patch.setattr(ops, "chain_prompt_takes", lambda *args, **sizes: False)  # (the same cache for all)
        if plan != "own":
            patch.setattr(ops, "chain_plan", lambda *args, **sizes: plan)
        engine = load_engine(folder, dtype="bfloat16", max_tokens=sum(-(-(n + 3) // 64) * 64 for n in lengths))
        engine.use_graphs = False  # (launched: what the final norm is handed is seen here)
        prompts, tokens = _tokens(lengths, 2)
        slots = [engine.start_sequence() for _ in lengths]
        engine.step([StepEntry(slot, prompt, None) for slot, prompt in zip(slots, prompts)])
        seen, norm = [], engine.model.final_norm
        add = norm.add_forward
        patch.setattr(norm, "add_forward", lambda x, delta, *args, **more: seen.extend((x.clone(), delta.clone())) or add(x, delta, *args, **more), raising=False)
        for row in tokens:
            engine.step([StepEntry(slot, [token], None) for slot, token in zip(slots, row)])
        chain = engine.model.layer_chain(engine.rt)
        return seen, chain is not None and len(chain.tables) > 0


# ... and whether the launch takes 3, 16 and 20 rows of them: the layers' kernels cut K in ways that it does not have
CUTS = [
    ((1024, 16, 4, 2048), (True, True, True)),
    ((1024, 17, 17, 512), (False, False, False)),   # the output projection in eight parts, four waves
    ((1024, 32, 8, 512), (False, False, False)),
    ((192, 6, 2, 5056), (True, True, True)),
    ((192, 6, 2, 5120), (False, False, True)),      # down by two blocks a strip, up to 16 rows
    ((2048, 31, 31, 1024), (True, True, False)),    # the runs' sum on the way into the output projection, up to four rows
    ((2048, 32, 32, 1024), (True, True, False)),    # ... and by a kernel of its own
    ((2048, 79, 79, 256), (True, True, False)),
    ((2048, 80, 20, 256), (False, False, False)),   # the output projection by two blocks a strip
    ((2112, 80, 20, 256), (True, True, False)),     # ... not above a width of 2,048
    ((3072, 24, 8, 8192), (True, True, False)),
    ((3072, 24, 8, 8256), (False, False, False)),   # gate and up in two parts
    ((4096, 64, 16, 4096), (True, True, False)),
]


@pytest.mark.parametrize("sizes, taken", CUTS)
def test_cuts_of_k(tmp_path, sizes, taken, monkeypatch):
    """Both sides of each line of ``chain_cuts_alike``: the stream's bits are the layers' kernels' wherever the launch is made."""
    import nnis_amd

    nnis_amd.write_random_model(str(tmp_path), _config(*sizes), 3)
    for batch, takes in zip((3, 16, 20), taken):
        lengths = (LENGTHS + [n + 1 for n in LENGTHS])[:batch] if batch != 3 else [1100, 1500, 700]
        layers, ran = _streams(str(tmp_path), lengths, None, monkeypatch)
        assert not ran
        got, ran = _streams(str(tmp_path), lengths, "own", monkeypatch)
        assert ran == takes, batch
        assert len(got) == 4 and all(torch.equal(a, b) for a, b in zip(got, layers)), batch


@pytest.mark.parametrize("sizes", [(2048, 31, 31, 1024), (2048, 32, 32, 1024), (3072, 24, 8, 8192), (1024, 16, 4, 2048)])
def test_a_single_rows_runs(tmp_path, sizes, monkeypatch):
    """A row alone, whose runs of keys the output projection's waves add up: the layers' bits on four waves and on eight, in four and eight
    parts of K, and where the layers round 32 heads' sums on their way in (two, four and eight runs)."""
    import nnis_amd
    from nnis_amd.kernels import ops

    nnis_amd.write_random_model(str(tmp_path), _config(*sizes), 3)
    for length in (1100, 2000, 3700):
        assert ops.decode_plan(1, sizes[2], length, width=sizes[1] * 64)[0] in (2, 4, 8)
        layers, ran = _streams(str(tmp_path), [length], None, monkeypatch)
        assert not ran
        got, ran = _streams(str(tmp_path), [length], "own", monkeypatch)
        assert ran and len(got) == 4 and all(torch.equal(a, b) for a, b in zip(got, layers)), length


@pytest.mark.parametrize("sizes, plans", [
    ((2048, 32, 4, 1024), ("own", (2, 8), (8, 8))),           # eight waves, 32 heads: in the output projection
    ((1024, 17, 17, 512), ((2, 4), (4, 4), (8, 4))),          # four waves and more than 16 heads: by a stage of its own
    ((1024, 32, 8, 512), ((2, 4), (4, 4), (8, 4))),
    ((1152, 33, 11, 576), ((2, 8), (8, 8))),                  # eight waves and more than 32
    ((192, 6, 1, 448), ("own", (8, 4), (16, 4))),             # up to eight runs, and more
])
def test_a_single_rows_runs_in_other_bits(tmp_path, sizes, plans, monkeypatch):
    """... and where the launch has bits of its own, as far from 32 bits as the layers' kernels (``test_against_the_layers``)."""
    import nnis_amd

    nnis_amd.write_random_model(str(tmp_path), _config(*sizes), 3)
    for length in (1100, 3700):
        want = _run(str(tmp_path), "float32", [length], None, monkeypatch)[0]
        layers = _run(str(tmp_path), "bfloat16", [length], None, monkeypatch)[0]
        for plan in plans:
            got, ran, _ = _run(str(tmp_path), "bfloat16", [length], plan, monkeypatch)
            assert ran and (got - want).norm() <= 1.33 * (layers - want).norm(), (length, plan)


@pytest.mark.parametrize("counts", [(2,), (16,), (33,), (177,), (600,), (1, 1, 15, 16, 1, 30, 33), (100, 3, 260, 2), (9,) * 20])
@pytest.mark.parametrize("sizes", SIZES + [(1088, 8, 8, 4160)])  # (eight waves with a second round of down's weights)
def test_prompts_against_the_layers(tmp_path, sizes, counts, monkeypatch):
    """As far from 32 bits as the layers' kernels, some rows of each prompt and the steps behind them (by the layers' kernels, from what
    the launch left in the cache); launched and replayed the same bits.  (The roundings are the same, the orders of the sums are not.)"""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry
    from nnis_amd.kernels import ops

    nnis_amd.write_random_model(str(tmp_path), _config(*sizes), 3)
    rng = np.random.default_rng(sum(counts))
    prompts, tokens = [rng.integers(0, 509, size=n).tolist() for n in counts], rng.integers(0, 509, size=2).tolist()
    places = [sorted({0, n // 3, n - 1}) for n in counts]

    def run(dtype, takes):
        with monkeypatch.context() as patch:
            launches = []
            launch = ops.chain_prompt
            patch.setattr(ops, "chain_prompt", lambda *args, **more: launches.append(1) or launch(*args, **more))
            if takes is not None:
                patch.setattr(ops, "chain_prompt_takes", lambda *args, **more: takes)
            patch.setattr(ops, "chain_plan", lambda *args, **more: None)
            engine = load_engine(str(tmp_path), dtype=dtype, max_tokens=2048)
            slots, out = [engine.start_sequence() for _ in counts], None
            for again in range(4):  # launched, launched and captured, replayed
                for slot in slots:
                    engine.truncate(slot, 0)
                got = [engine.step([StepEntry(*entry) for entry in zip(slots, prompts, places)]).double().cpu()]
                for token in tokens:
                    got.append(engine.step([StepEntry(slot, [token], None) for slot in slots]).double().cpu())
                got = torch.cat(got)
                assert dtype == "float32" or not launches or out is None or torch.equal(out, got)
                out = got
            return out, len(launches)

    want, _ = run("float32", None)
    layers, launched = run("bfloat16", False)
    assert launched == 0
    got, launched = run("bfloat16", True)
    assert launched > 0
    error, bound = (got - want).norm(), 1.33 * (layers - want).norm()
    assert error <= bound, f"{error.item():.4g} from 32 bits, the layers' kernels {(layers - want).norm().item():.4g}"


def test_prompts_that_are_not_taken(tmp_path, monkeypatch):
    """A prompt behind cached tokens, also beside one that begins, and one beyond the rows: the layers' kernels, also where a prompt of
    the same rows has been captured."""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry
    from nnis_amd.kernels import ops

    nnis_amd.write_random_model(str(tmp_path), _config(192, 6, 2, 1600), 3)
    launches = []
    launch = ops.chain_prompt
    monkeypatch.setattr(ops, "chain_prompt", lambda *args, **more: launches.append(1) or launch(*args, **more))
    engine = load_engine(str(tmp_path), dtype="bfloat16", max_tokens=4096)
    plain = load_engine(str(tmp_path), dtype="float32", max_tokens=4096)
    rng = np.random.default_rng(5)
    first, second = rng.integers(0, 509, size=40).tolist(), rng.integers(0, 509, size=50).tolist()
    slot, other = engine.start_sequence(), plain.start_sequence()
    for _ in range(3):
        engine.truncate(slot, 0)
        engine.step([StepEntry(slot, second, None)])
    taken = len(launches)
    assert taken > 0
    engine.truncate(slot, 0)
    engine.step([StepEntry(slot, first, None)])
    plain.step([StepEntry(other, first, None)])
    taken = len(launches)
    for _ in range(3):  # the same 64 rows as the captured prompt's
        engine.truncate(slot, len(first))
        plain.truncate(other, len(first))
        got, want = engine.step([StepEntry(slot, second, None)]), plain.step([StepEntry(other, second, None)])
        assert (got.double() - want.double()).norm() <= 0.05 * want.double().norm()  # (a few bfloat16 roundings of 2^-9 over two layers)
    assert len(launches) == taken
    engine.truncate(slot, 7)
    engine.step([StepEntry(engine.start_sequence(), first, None), StepEntry(slot, first, None)])
    engine.step([StepEntry(engine.start_sequence(), rng.integers(0, 509, size=1100).tolist(), None)])
    assert len(launches) == taken


def test_prompts_in_a_step_do_not_meet(tmp_path):
    """What a sequence holds that is not finite stays its own: the others' logits are the same bits as beside finite ones."""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry

    nnis_amd.write_random_model(str(tmp_path), dict(_config(192, 6, 2, 1600), tie_word_embeddings=False), 3)
    engine = load_engine(str(tmp_path), dtype="bfloat16", max_tokens=2048)
    rng = np.random.default_rng(7)
    prompts = [rng.integers(8, 509, size=n).tolist() for n in (5, 20, 3, 40, 17)]
    prompts[1][9] = prompts[3][0] = 7
    slots = [engine.start_sequence() for _ in prompts]

    def step():
        for slot in slots:
            engine.truncate(slot, 0)
        return engine.step([StepEntry(slot, prompt, None) for slot, prompt in zip(slots, prompts)])

    finite = step()
    table = engine.model.embedding.table
    table[7] = float("inf")
    for _ in range(3):
        got = step()
        assert torch.equal(got[[0, 2, 4]], finite[[0, 2, 4]]) and not bool(torch.isfinite(got[[1, 3]]).any())


def test_not_taken(tmp_path, monkeypatch):
    """Other head sizes and sizes in other steps than 64 stay with the layers' kernels."""
    import nnis_amd

    for index, change in enumerate(({"head_dim": 32}, {"intermediate_size": 176})):
        folder = tmp_path / str(index)
        folder.mkdir()
        nnis_amd.write_random_model(str(folder), dict(_config(64, 1, 1, 64), **change), 3)
        for dtype in ("bfloat16", "float32"):
            assert not _run(str(folder), dtype, [40], "own", monkeypatch)[1]


def test_a_wait_given_up_is_reported(tmp_path, monkeypatch):
    """The word that a kernel writes when it gives a wait up (written here by the host) refuses the next step, and the sequence until it
    has been emptied."""
    import nnis_amd
    from nnis_amd.engine.batch import StepEntry

    nnis_amd.write_random_model(str(tmp_path), _config(64, 1, 1, 64), 3)
    _, ran, engine = _run(str(tmp_path), "bfloat16", [40], "own", monkeypatch)
    assert ran
    slot = next(iter(engine.cache.lengths))
    length = engine.length(slot)
    engine.model.layer_chain(engine.rt).failed[0] = 1
    with pytest.raises(KernelError, match="gave up waiting"):
        engine.step([StepEntry(slot, [7], None)])
    assert engine.length(slot) == length
    with pytest.raises(KernelError, match="not numbers"):
        engine.step([StepEntry(slot, [7], None)])
    engine.truncate(slot, 0)
    assert bool(torch.isfinite(engine.step([StepEntry(slot, [7], None)])).all())
    engine.use_graphs = False  # launched, not replayed
    engine.model.layer_chain(engine.rt).failed[0] = 1
    with pytest.raises(KernelError, match="gave up waiting"):
        engine.step([StepEntry(slot, [7], None)])
    assert engine.length(slot) == 1


def test_sequences_of_a_lost_step(tmp_path):
    """Those that were in it are refused until they end, and leave no NaN to whoever takes their pages; the others, and those whose last step
    is known to have ended well, go on with the same bits."""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry
    from nnis_amd.sampling.device import DeviceSelector

    nnis_amd.write_random_model(str(tmp_path), _config(64, 1, 1, 64), 3)
    engine = load_engine(str(tmp_path), dtype="bfloat16", max_tokens=320)
    selector = DeviceSelector(engine)
    first, second, third = (engine.start_sequence() for _ in range(3))
    prompts = {first: [1, 2, 3], second: list(range(70)), third: [9, 8]}

    def step(slots, tokens):
        logits = engine.step([StepEntry(slot, tokens[slot], None) for slot in slots])
        return logits, selector.select_start(logits, slots, [None] * len(slots))

    step([first, second, third], prompts)[1].result()  # (known to have ended well)
    want, _ = step([first], {first: [5]})
    engine.truncate(first, 3)
    selector.select_start(want, [first], [None]).result()
    _, lost = step([second, third], {second: [5], third: [6]})
    engine.model.layer_chain(engine.rt).failed[0] = 1
    for view in (engine.cache.view(0), engine.cache.view(1)):  # what such a step leaves, also in pages that have gone back since
        for slot in (second, third):
            for page in engine.cache.kv_groups[0].table.rows[slot]:
                view.k_pages[page] = view.v_pages[page] = float("nan")
    engine.end_sequence(third)
    with pytest.raises(StepLost):
        lost.result()
    assert torch.equal(step([first], {first: [5]})[0], want)
    with pytest.raises(StepLost, match="not numbers"):
        engine.step([StepEntry(second, [5], None)])
    with pytest.raises(StepLost, match="not numbers"):
        engine.step([StepEntry(first, [5], None), StepEntry(second, [5], None)])
    assert engine.length(first) == 4 and engine.length(second) == 71
    engine.end_sequence(second)
    for _ in range(2):  # (two pages each of the four that are free: those of the lost step among them)
        slot = engine.start_sequence()
        engine.step([StepEntry(slot, list(range(65)), None)])
        assert bool(torch.isfinite(engine.step([StepEntry(slot, [5], None)])).all())
    for view in (engine.cache.view(0), engine.cache.view(1)):
        assert bool(torch.isfinite(view.k_pages).all()) and bool(torch.isfinite(view.v_pages).all())


def test_a_report_is_no_refusal(tmp_path):
    """The report reaches the caller also at the step with which a shape of prompts would be captured, and the shape is captured later."""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry

    nnis_amd.write_random_model(str(tmp_path), _config(64, 1, 1, 64), 3)
    engine = load_engine(str(tmp_path), dtype="bfloat16", max_tokens=512)
    prompt = list(range(20))

    def step():
        return engine.step([StepEntry(engine.start_sequence(), prompt, None)])

    want = step()
    engine.model.layer_chain(engine.rt).failed[0] = 1
    with pytest.raises(StepLost, match="gave up waiting"):
        step()
    for _ in range(3):
        assert torch.equal(step(), want)
    assert len(engine._prefill_graphs.graphs) == 1 and not engine._prefill_graphs.refused


def _lose(engine, call, at):
    """Patches ``engine`` so that the ``at``-th step's launch is followed by the word that a given-up wait writes."""
    count = [0]

    def wrap(step):
        def run(*args):
            out = step(*args)
            count[0] += 1
            if count[0] == at:
                engine.model.layer_chain(engine.rt).failed[0] = 1
            return out
        return run

    for name in ("step_view", "step_from_device"):
        call.setattr(engine, name, wrap(getattr(engine, name)))


@pytest.mark.parametrize("new, at", [(1, 1), (6, 1), (6, 3), (6, 6)])
@pytest.mark.parametrize("ahead", [True, False])
def test_tokens_of_a_lost_step_go_nowhere(tmp_path, new, at, ahead, monkeypatch):
    """A request whose step gave a wait up, its only one, its first, a later one or its last, gets an error and no token of that step; the
    next request gets its tokens."""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.generate import GenerationRequest, generate

    nnis_amd.write_random_model(str(tmp_path), _config(64, 1, 1, 64), 3)
    engine = load_engine(str(tmp_path), dtype="bfloat16", max_tokens=512)
    engine.use_graphs = ahead
    prompts = [list(range(20)), list(range(30, 37))]
    seen = [[], []]
    want = [r.tokens for r in generate(engine, [GenerationRequest(p, new) for p in prompts])]
    with monkeypatch.context() as patch:
        _lose(engine, patch, at)
        with pytest.raises(StepLost, match="gave up waiting"):
            generate(engine, [GenerationRequest(p, new, on_token=lambda i, token: seen[i].append(token) or True) for p in prompts])
    for tokens, right in zip(seen, want):
        assert tokens == right[:len(tokens)] and len(tokens) < at
    assert not engine.cache.lengths
    assert [r.tokens for r in generate(engine, [GenerationRequest(p, new) for p in prompts])] == want


def test_pending_tokens_of_a_lost_step(tmp_path):
    """Written between the selection and its result."""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry
    from nnis_amd.sampling.device import DeviceSelector

    nnis_amd.write_random_model(str(tmp_path), _config(64, 1, 1, 64), 3)
    engine = load_engine(str(tmp_path), dtype="bfloat16", max_tokens=512)
    selector = DeviceSelector(engine)
    slot = engine.start_sequence()
    pending = selector.select_start(engine.step_view([StepEntry(slot, [1, 2, 3], None)]), [slot], [None])
    engine.model.layer_chain(engine.rt).failed[0] = 1
    with pytest.raises(StepLost):
        pending.result()


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("sizes", [(192, 6, 2, 192), (1088, 8, 8, 576)])
def test_what_lies_behind_a_sequence_does_not_matter(tmp_path, sizes, dtype, monkeypatch):
    """Keys and values from the step's own place in a page on may be no numbers: the same bits as over zeros."""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry

    nnis_amd.write_random_model(str(tmp_path), _config(*sizes), 3)
    engine = load_engine(str(tmp_path), dtype=dtype, max_tokens=4096)
    lengths = [1, 7, 8, 31, 32, 40, 62, 63, 64, 65, 100, 1100]
    prompts, tokens = _tokens(lengths, 1)
    slots = [engine.start_sequence() for _ in lengths]
    for slot, prompt in zip(slots, prompts):
        engine.step([StepEntry(slot, prompt, None)])

    def step(fill):
        for slot, n in zip(slots, lengths):
            engine.truncate(slot, n)
            row = engine.cache.kv_groups[0].table.rows[slot]
            for index in range(2) if n % 64 else ():
                view = engine.cache.view(index)
                for t in range(n % 64, 64):
                    view.k_pages[row[-1]][:, :, t] = fill
                    view.v_pages[row[-1]][:, :, t // 32, t % 32 // 8, :, t % 8] = fill
        return engine.step([StepEntry(slot, [token], None) for slot, token in zip(slots, tokens[0])])

    want = step(0.0)
    assert len(engine.model.layer_chain(engine.rt).tables) > 0
    for fill in (float("nan"), float("inf")):
        assert torch.equal(step(fill), want)


def test_one_exchange_for_all_shapes(tmp_path):
    """Steps of any shape, launched and captured, share the exchange: captured shapes do not add up. A larger shape gets a larger one, and
    graphs go on with the one that they were captured with."""
    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry

    nnis_amd.write_random_model(str(tmp_path), _config(576, 9, 3, 1536, layers=6), 3)
    engine = load_engine(str(tmp_path), dtype="bfloat16", max_tokens=2048)
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, 509, size=n).tolist() for n in (40, 1000, 100, 200, 400, 700)]

    def step(prompt):
        slot = engine.start_sequence()
        out = [engine.step([StepEntry(slot, prompt, None)]), engine.step([StepEntry(slot, [7], None)])]
        engine.end_sequence(slot)
        return torch.cat(out)

    want = [step(prompt) for prompt in prompts]
    chain = engine.model.layer_chain(engine.rt)
    largest = chain.exchange
    words, needed = [], nnis_amd.kernels.ops.chain_module().nnis_chain_prompt_words(6, 1024, 576, 9, 3, 1536)
    assert needed <= largest.numel() <= 2 * needed
    for _ in range(3):  # captured, replayed; the shapes in turn
        for prompt, first in zip(prompts, want):
            assert torch.equal(step(prompt), first)
            words.append(chain.exchange)
    graphs = list(engine._prefill_graphs.graphs.values())
    assert len(graphs) == len(prompts) and all(word is largest for word in words)
    assert all(any(buffer is largest for buffer in graph.held_of_launches) for graph in graphs)


@pytest.mark.parametrize("lengths", [(150, 90, 33), (700, 570, 950)])  # (keys in one run, and in several in the scratch that all have)
@pytest.mark.parametrize("threads", [False, True])
def test_launches_on_two_streams_take_turns(tmp_path, threads, lengths):
    """Two engines on streams of their own, over one model and over two, from one thread and from two: neither waits for what the other's
    launch keeps off the chip, and each has the bits that it has alone."""
    import threading

    import nnis_amd
    from nnis_amd.api import load_engine
    from nnis_amd.engine.batch import StepEntry
    from nnis_amd.engine.step import Engine

    nnis_amd.write_random_model(str(tmp_path), _config(576, 9, 3, 1536, layers=8), 3)
    first, other = (load_engine(str(tmp_path), dtype="bfloat16", max_tokens=1024) for _ in range(2))
    engines = [first, Engine(first.model, first.rt, max_tokens=1024), other]
    rng = np.random.default_rng(11)
    prompts = [rng.integers(0, 509, size=n).tolist() for n in lengths]

    def steps(engine, prompt):
        slot, out = engine.start_sequence(), []
        for number in range(25):
            if number % 8 == 0:  # (launched, captured, replayed)
                engine.truncate(slot, 0)
                out.append(engine.step([StepEntry(slot, prompt, None)]))
            out.append(engine.step([StepEntry(slot, [number], None)]))
            yield
        engine.end_sequence(slot)
        yield torch.cat(out)

    def alone(engine, prompt):
        *_, out = steps(engine, prompt)
        return out

    want = [alone(engine, prompt) for engine, prompt in zip(engines, prompts)]
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream() for _ in engines], [None] * len(engines)
    if threads:
        def run(index):
            with torch.cuda.stream(streams[index]):
                got[index] = alone(engines[index], prompts[index])

        workers = [threading.Thread(target=run, args=(index,)) for index in range(len(engines))]
        for worker in workers:
            worker.start()
        for worker in workers:
            worker.join()
    else:
        runs = [steps(engine, prompt) for engine, prompt in zip(engines, prompts)]
        for _ in range(26):
            for index, run in enumerate(runs):
                with torch.cuda.stream(streams[index]):
                    got[index] = next(run)
    torch.cuda.synchronize()
    for engine, a, b in zip(engines, got, want):
        assert torch.equal(a, b)
        engine.check_steps()


def test_sizes_and_words():
    """The exchange's size is 0 for what the launch refuses, and grows with what it holds."""
    from nnis_amd.kernels import ops

    words = ops.chain_words
    assert words(2, 1, 64, 1, 1, 64, 1)[0] > 0 and words(2, 1, 64, 1, 1, 64, 1)[1] == 0
    assert words(2, 2, 64, 1, 1, 64, 1)[0] > words(2, 1, 64, 1, 1, 64, 1)[0] and words(2, 2, 64, 1, 1, 64, 2)[1] == 2 * 2 * 2 * 68
    for refused in ((2, 33, 64, 1, 1, 64, 1), (2, 17, 1088, 1, 1, 64, 1), (2, 0, 64, 1, 1, 64, 1), (2, 1, 96, 1, 1, 64, 1), (2, 1, 64, 3, 2, 64, 1), (2, 1, 64, 1, 1, 80, 1),
                    (2, 1, 64, 1, 1, 64, 17), (0, 1, 64, 1, 1, 64, 1)):
        assert words(*refused)[0] == 0 and words(*refused, torch.float32)[0] == 0
    assert words(2, 1, 64, 16, 1, 64, 1, torch.float32)[0] > 0 and words(2, 1, 64, 17, 1, 64, 1, torch.float32)[0] == 0
