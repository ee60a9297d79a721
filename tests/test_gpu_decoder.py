"""The decoder language models through the engine on the device: prompts, decoding, portions, sequences, generation and the
command line, against the plain implementation, on small models of several shapes."""
import importlib
import json
import os
import subprocess

import numpy as np
import pytest

import decoder_cases as cases
import decoder_oracle as plain

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIMIT = {True: 3e-5, False: 6e-2}        # of the logits' spread; bf16: a planted mistake moves them by more


@pytest.fixture(scope="module")
def decoder():
    return importlib.import_module("qingming-qwen3-tts_amd.decoder")


class Model:
    def __init__(self, name, directory, count):
        self.cfg = cases.CONFIGS[name]
        self.weights = cases.weights(self.cfg)
        self.directory = str(directory)
        cases.write_model(self.directory, self.cfg, self.weights)
        self.tokens = cases.tokens_of(self.cfg, count)
        self.streams = []
        self.want = plain.forward(self.cfg, self.weights, self.tokens, self.streams)


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    made = {}

    def make(name, count=170):
        if name not in made:
            made[name] = Model(name, tmp_path_factory.mktemp(name), count)
        return made[name]
    return make


def feed(engine, sequence, tokens, portions):
    """Logits of every position, the tokens fed in these portions."""
    got, at = [], 0
    for n in portions:
        got.append(engine.step(sequence, tokens[at:at + n], np.arange(n)))
        at += n
    assert at == len(tokens)
    return np.concatenate(got)


NAMES = sorted(cases.CONFIGS)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("name", NAMES)
def test_prompt_and_streams(decoder, models, name, f32):
    m = models(name)
    engine = decoder.Decoder(m.directory, len(m.tokens), float32=f32)
    s = engine.open()
    logits, streams = engine.step(s, m.tokens, np.arange(len(m.tokens)), streams=True)
    assert cases.error(logits, m.want) < LIMIT[f32]
    for i, want in enumerate(m.streams):
        assert cases.error(streams[i], want) < LIMIT[f32], i
    assert engine.runs == len(m.streams) == len(plain.layer_runs(m.cfg))


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("name", NAMES)
def test_portions_decoding_and_reuse(decoder, models, name, f32):
    """One engine, its one sequence used again and again: every way of cutting gives the same logits."""
    m = models(name)
    n = len(m.tokens)
    engine = decoder.Decoder(m.directory, n, float32=f32)
    cuts = ([1] * n, [n - 40] + [1] * 40, [2] * (n // 2), [3, 1, 16, 15, 1, 1, 17, 33, 5, 64, n - 156], [n])
    for path in (0, 1, 2, 4):
        engine.set_path(path)
        for portions in cuts if path == 0 else cuts[1:4:2]:
            s = engine.open()
            got = feed(engine, s, m.tokens, portions)
            engine.close(s)
            assert cases.error(got, m.want) < LIMIT[f32], (path, portions)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("name", NAMES)
def test_sequences_side_by_side(decoder, models, name, f32):
    """Two sequences in turn, one of them closed and its memory used again by a third: none notices the others."""
    m = models(name)
    other = cases.tokens_of(m.cfg, len(m.tokens), seed=7)
    want_other = plain.forward(m.cfg, m.weights, other)
    engine = decoder.Decoder(m.directory, len(m.tokens), float32=f32, sequences=2)
    a, b = engine.open(), engine.open()
    with pytest.raises(decoder.DecoderError) as e:
        engine.open()
    assert e.value.code == -3
    got_a, got_b, at_a, at_b = [], [], 0, 0
    for n_a, n_b in ((40, 3), (1, 60), (1, 1), (1, 1), (1, 1), (17, 2), (1, 1)):
        got_a.append(engine.step(a, m.tokens[at_a:at_a + n_a], np.arange(n_a)))
        got_b.append(engine.step(b, other[at_b:at_b + n_b], np.arange(n_b)))
        at_a, at_b = at_a + n_a, at_b + n_b
    assert cases.error(np.concatenate(got_a), m.want[:at_a]) < LIMIT[f32]
    assert cases.error(np.concatenate(got_b), want_other[:at_b]) < LIMIT[f32]
    engine.close(b)
    c = engine.open()
    assert cases.error(feed(engine, c, m.tokens[:60], [20, 1, 1, 1, 37]), m.want[:60]) < LIMIT[f32]
    assert cases.error(engine.step(a, m.tokens[at_a:at_a + 1], [0]), m.want[at_a:at_a + 1]) < LIMIT[f32]


@pytest.mark.parametrize("f32", [True, False])
def test_passes_of_few_rows_and_small_rings(decoder, models, f32):
    """A prompt longer than a pass, in an engine whose rings are a few positions longer than the chunks."""
    for name, capacity in (("short_chunks", 100000), ("mixed", 300), ("retention", 100000)):
        m = models(name)
        for max_rows in (3, 20, 64):
            engine = decoder.Decoder(m.directory, capacity, float32=f32, max_rows=max_rows)
            assert engine.sequence_bytes < 2 ** 20
            s = engine.open()
            assert cases.error(feed(engine, s, m.tokens, [120] + [1] * 20 + [30]), m.want) < LIMIT[f32]


@pytest.mark.parametrize("name", ["short_chunks", "looped", "mixed", "latents"])
def test_long_decoding(decoder, models, name):
    m = models(name)
    tokens = cases.tokens_of(m.cfg, 420, seed=3)
    want = plain.forward(m.cfg, m.weights, tokens)
    for f32 in (True, False):
        engine = decoder.Decoder(m.directory, 420, float32=f32, max_rows=32)
        s = engine.open()
        assert cases.error(feed(engine, s, tokens, [20] + [1] * 400), want) < LIMIT[f32]


def test_wanted_places_in_any_order(decoder, models):
    m = models("plain")
    engine = decoder.Decoder(m.directory, len(m.tokens), float32=True, max_rows=50)
    want = [160, 3, 3, 99, 49, 50, 0]
    got = engine.step(engine.open(), m.tokens, want)
    assert cases.error(got, m.want[want]) < LIMIT[True]
    engine = decoder.Decoder(m.directory, len(m.tokens), float32=True)
    assert engine.step(engine.open(), m.tokens[:5]).shape == (0, m.cfg["vocab"])


@pytest.mark.parametrize("name", ["plain", "mixed"])
def test_ways_of_stepping_leave_the_same(decoder, models, name):
    """Steps whose scores come through pinned memory, steps that want none, several copies, queued steps and generation in turn, two
    sequences of one engine: the scores of every token are those of plain fused launches, bit for bit (77 scores: no multiple of four)."""
    m = models(name)
    tokens = m.tokens[:40]
    plain_engine = decoder.Decoder(m.directory, len(m.tokens), sequences=2)
    plain_engine.set_path(1)
    p = plain_engine.open()
    want = [plain_engine.step(p, tokens[:9], [8])[0]] + [plain_engine.step(p, [t], [0])[0] for t in tokens[9:]]
    engine = decoder.Decoder(m.directory, len(m.tokens), sequences=2)
    a, b = engine.open(), engine.open()
    for s in (a, b):
        assert np.array_equal(engine.step(s, tokens[:9], [8])[0], want[0])
    for i, t in enumerate(tokens[9:], 1):
        for s in (a, b):
            if (i + s) % 4 == 0:
                engine.step(s, [t])
            elif (i + s) % 4 == 1:
                engine.enqueue(s, [t])
            else:
                got = engine.step(s, [t], [0] * (i % 3 + 1))
                assert got.shape[0] == i % 3 + 1 and all(np.array_equal(row, want[i]) for row in got)
    made = engine.generate(a, [int(tokens[0])], 5)
    assert np.array_equal(made, plain_engine.generate(p, [int(tokens[0])], 5))
    assert np.array_equal(engine.step(a, [1], [0]), plain_engine.step(p, [1], [0]))


@pytest.mark.parametrize("vocab", [2047, 2049, 5122, 16384 + 3])
def test_scores_of_large_vocabularies_through_pinned_memory(decoder, tmp_path, vocab):
    """One block, two, five and sixteen write a step's scores, each raising a flag of its own, the last vocabulary's remainder by the first:
    every score is the plain launches', bit for bit, and none the step before's."""
    cfg = cases.config(vocab, 64, [cases.general_delta(2, 16, 32)])
    cases.write_model(str(tmp_path), cfg, cases.weights(cfg))
    tokens = cases.tokens_of(cfg, 40)
    rows = []
    for path in (1, 0):
        engine = decoder.Decoder(str(tmp_path), 64)
        engine.set_path(path)
        s = engine.open()
        rows.append([engine.step(s, tokens[:7], [6])[0]] + [engine.step(s, [t], [0])[0] for t in tokens[7:]])
    for i, (want, got) in enumerate(zip(*rows)):
        assert np.array_equal(got, want), i
        assert i == 0 or (got != rows[1][i - 1]).mean() > 0.9


def test_steps_behind_long_work(decoder, models, dev):
    """Scores that tens of milliseconds of other work on the stream are ahead of: waited for, and the step's own."""
    import torch
    m = models("plain")
    stream = torch.cuda.Stream()
    engine = decoder.Decoder(m.directory, len(m.tokens), stream=stream.cuda_stream)

    def run(before):
        s = engine.open()
        got = []
        for tokens in (m.tokens[:9], m.tokens[9:10], m.tokens[10:11]):
            before()
            got.append(engine.step(s, tokens, [len(tokens) - 1])[0])
        engine.close(s)
        return got

    a = torch.ones(4096, 4096, device=dev)
    torch.cuda.synchronize()

    def work():
        with torch.cuda.stream(stream):
            for _ in range(80):
                a @ a

    for got, want in zip(run(work), run(lambda: None)):
        assert np.array_equal(got, want)


def greedy(m, prompt, count):
    tokens = list(prompt)
    for _ in range(count):
        tokens.append(int(plain.forward(m.cfg, m.weights, tokens)[-1].argmax()))
    return tokens[len(prompt):]


@pytest.mark.parametrize("name", NAMES)
def test_greedy_generation(decoder, models, name):
    m = models(name)
    prompt = m.tokens[:23]
    want = greedy(m, prompt, 24)
    engine = decoder.Decoder(m.directory, 64, float32=True)
    for path in (0, 1, 2):
        engine.set_path(path)
        s = engine.open()
        assert list(engine.generate(s, prompt, 24)) == want
        engine.close(s)
    stop = want[9]
    s = engine.open()
    assert list(engine.generate(s, prompt, 24, stop_token=stop)) == want[:want.index(stop) + 1]
    engine.close(s)
    s = engine.open()                                            # a prompt of one token; a sequence that goes on
    first = engine.generate(s, prompt[:1], 3)
    assert list(first) == greedy(m, prompt[:1], 3)
    more = engine.generate(s, [first[-1]], 4)
    assert list(more) == greedy(m, list(prompt[:1]) + list(first), 4)


def test_sampled_generation_is_the_samplers(decoder, models):
    """top_k = 1 is the arg-max; a seed gives its own tokens again, all of them among the k most likely."""
    m = models("plain")
    engine = decoder.Decoder(m.directory, 80, float32=True)

    def run(**options):
        s = engine.open()
        out = list(engine.generate(s, m.tokens[:20], 30, **options))
        engine.close(s)
        return out

    assert run(top_k=1, temperature=0.7, seed=5) == run()
    a, b = run(top_k=8, temperature=1.0, seed=5), run(top_k=8, temperature=1.0, seed=6)
    assert a == run(top_k=8, temperature=1.0, seed=5) and a != b
    logits = plain.forward(m.cfg, m.weights, list(m.tokens[:20]) + a)
    for i, token in enumerate(a):
        assert token in np.argsort(-logits[19 + i])[:8]


def test_errors_leave_the_engine_usable(decoder, models):
    m = models("plain")
    engine = decoder.Decoder(m.directory, 40, float32=True)
    s = engine.open()
    for bad in (lambda: engine.step(s, []), lambda: engine.step(s, [m.cfg["vocab"]]), lambda: engine.step(s, [-1]), lambda: engine.step(s, m.tokens[:41]),
                lambda: engine.step(s, m.tokens[:4], [4]), lambda: engine.step(s + 1, m.tokens[:4]), lambda: engine.generate(s, m.tokens[:20], 22),
                lambda: engine.generate(s, m.tokens[:4], 4, top_k=300), lambda: engine.set_path(3)):
        with pytest.raises(decoder.DecoderError):
            bad()
    assert cases.error(feed(engine, s, m.tokens[:40], [39, 1]), m.want[:40]) < LIMIT[True]
    with pytest.raises(decoder.DecoderError):
        engine.step(s, [1])
    engine.close(s)
    with pytest.raises(decoder.DecoderError):
        engine.step(s, [1])


@pytest.mark.parametrize("model,name", [("plain", "l1.mix.w2"), ("mixed", "l2.mlp.e11.up"), ("mixed", "l0.mix.dkv"), ("retention", "bigram")])
@pytest.mark.parametrize("change,code", [("missing", -8), ("shape", -8), ("dtype", -8)])
def test_wrong_weights_are_refused(decoder, tmp_path, change, code, model, name):
    import torch
    from safetensors.torch import load_file, save_file
    cfg = cases.CONFIGS[model]
    cases.write_model(str(tmp_path), cfg, cases.weights(cfg))
    path = os.path.join(str(tmp_path), "model.safetensors")
    tensors = load_file(path)
    if change == "missing":
        del tensors[name]
    elif change == "shape":
        tensors[name] = tensors[name][:-1].contiguous()
    else:
        tensors[name] = tensors[name].to(torch.float32)
    save_file(tensors, path)
    with pytest.raises(decoder.DecoderError) as e:
        decoder.Decoder(str(tmp_path), 16)
    assert e.value.code == code and name in str(e.value)


def test_first_tokens_and_the_token_before(decoder, models):
    """A sequence's first token has none before it, also in memory that was used; the next step's first token has the last one's."""
    m = models("retention")
    engine = decoder.Decoder(m.directory, 64, float32=True)
    for portions in ([1, 1, 1, 1], [2, 2], [1, 3], [3, 1], [4]):
        s = engine.open()
        assert cases.error(feed(engine, s, m.tokens[:4], portions), m.want[:4]) < LIMIT[True]
        engine.generate(s, m.tokens[4:9], 3)
        engine.close(s)
    engine.set_path(2)
    s = engine.open()
    assert cases.error(feed(engine, s, m.tokens[:6], [1, 1, 3, 1]), m.want[:6]) < LIMIT[True]


@pytest.mark.parametrize("f32", [True, False])
def test_a_far_key_decides(decoder, tmp_path, f32):
    """Latent attention whose query looks for one token: its only occurrence is hundreds of positions back, at a pass's edge or in the
    middle, and the logits tell it from a sequence without it."""
    cfg = cases.sandwich(48, 96, [cases.latent(4, 24, 8, 32, 40, 64, cases.dense(64))], (13, 3, 1), residual_mult=2.0)
    w = cases.weights(cfg, seed=3)
    # token 7's latent stands out: a direction of its own through dkv and up_k, which every query carries through dq and up_q
    rng = np.random.default_rng(4)
    mark, mark_c, mark_q = (cases.bf16(v / np.linalg.norm(v)) for v in (rng.standard_normal(96), rng.standard_normal(64), rng.standard_normal(40)))
    w["embed"][7] = cases.bf16(60 * mark)
    w["l0.mix.dkv"][:64] = cases.bf16(0.3 * w["l0.mix.dkv"][:64] + 2.0 * np.outer(mark_c, mark))
    head = cases.bf16(np.ones(24) * 0.4)
    for h in range(4):
        w["l0.mix.uk"][24 * h:24 * h + 24] = cases.bf16(0.1 * w["l0.mix.uk"][24 * h:24 * h + 24] + 4.0 * np.outer(head, mark_c))
        w["l0.mix.uq"][32 * h:32 * h + 24] = cases.bf16(0.1 * w["l0.mix.uq"][32 * h:32 * h + 24] + 6.0 * np.outer(head, mark_q))
    cases.write_model(str(tmp_path), cfg, w)
    tokens = cases.tokens_of(cfg, 700, seed=2)
    tokens[tokens == 7] = 8
    for at in (0, 63, 64, 65, 127, 300, 511, 639):
        marked = tokens.copy()
        marked[at] = 7
        want = plain.forward(cfg, w, marked)
        if at == 0:
            # (half of the queries look for the mark, the others away from it)
            moved = np.abs(want - plain.forward(cfg, w, tokens)).max(axis=1)[650:] / np.abs(want).max()
            assert np.quantile(moved, 0.75) > 0.1
        engine = decoder.Decoder(str(tmp_path), 700, float32=f32)
        for portions in ([660] + [1] * 40, [at + 1, 699 - at], [64, 2, 62, 572]):
            s = engine.open()
            got = feed(engine, s, marked, portions)
            engine.close(s)
            assert cases.error(got[640:], want[640:]) < LIMIT[f32], (at, portions)


def test_trace_replay_program(models, tmp_path):
    m = models("looped")
    lines, at = [], {"a": 0, "b": 0}
    wanted = []
    for step, (name, n, want) in enumerate([("a", 60, [0, 59]), ("a", 1, [0]), ("a", 2, []), ("b", 30, [29]), ("b", 1, [0]), ("a", 25, [3, 24])]):
        tokens = m.tokens[at[name]:at[name] + n]
        end = ["a", "b"] if step == 5 else []
        lines.append(json.dumps({"step": step, "entries": [{"id": name, "tokens": [int(t) for t in tokens], "want": want}], "end": end}))
        wanted.append([at[name] + w for w in want])
        at[name] += n
    p = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", m.directory, "--dtype", "float32", "--out", str(tmp_path), "--max-tokens", "200"],
                       input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stderr
    assert [line for line in p.stdout.splitlines() if line.startswith("done")] == [f"done {i}" for i in range(6)]
    for step, places in enumerate(wanted):
        path = os.path.join(str(tmp_path), f"{step}.f32")
        assert os.path.exists(path) == bool(places)
        if places:
            got = np.fromfile(path, "<f4").reshape(len(places), -1)
            assert cases.error(got, m.want[places]) < LIMIT[True]


def test_generate_program(decoder, models):
    m = models("plain")
    prompts = [[int(t) for t in m.tokens[:9]], [int(t) for t in m.tokens[5:30]]]
    p = subprocess.run([os.path.join(ROOT, "bin", "generate"), "--model", m.directory, "--dtype", "float32", "--max-new", "6"],
                       input="\n".join(map(json.dumps, prompts)) + "\n", capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stderr
    assert [json.loads(line) for line in p.stdout.splitlines()] == [greedy(m, prompt, 6) for prompt in prompts]


@pytest.mark.parametrize("float32", [False, True])
@pytest.mark.parametrize("design", ["parallel", "sandwich", "looped"])
def test_weights_beyond_the_cache_give_the_same_bits(decoder, tmp_path, design, float32):
    """A model whose head alone is more than the last-level cache keeps reads a step's weights with the non-temporal hint: the small model's scores, bit for
    bit (the large vocabulary's rows repeat the small one's)."""
    small, times = 1000, 1100                                  # 1 100 000 x 128 values of two bytes: 268 MiB
    if design != "sandwich":
        layers = [cases.parallel(cases.left(4, 2, 32, 48, 40, 16), cases.right(2, 32, 64, [0.9, 0.99]), 300), cases.general_delta(2, 32, 200)]
        make = lambda vocab: cases.config(vocab, 128, layers, loop=(0, 1, 3) if design == "looped" else None)
    else:
        layers = [cases.latent(4, 16, 8, 24, 48, 40, cases.moe(6, 2, 48)), cases.retention(2, 16, 24, [0.9, 0.99], cases.dense(300))]
        make = lambda vocab: cases.sandwich(vocab, 128, layers, (11, 6, 7))
    weights = cases.weights(make(small))
    tokens = cases.tokens_of(make(small), 30)
    rows = []
    for count in (1, times):
        where = tmp_path / str(count)
        where.mkdir()
        cases.write_model(str(where), make(small * count), {name: np.tile(w, (count, 1)) if name in ("embed", "head") else w for name, w in weights.items()})
        engine = decoder.Decoder(str(where), 32, float32=float32)
        s = engine.open()
        rows.append([engine.step(s, tokens[:5], [4])[0]] + [engine.step(s, [t], [0])[0] for t in tokens[5:]])
        engine.close(s)
        del engine
    for want, got in zip(*rows):
        assert np.array_equal(got, np.tile(want, times))


@pytest.mark.parametrize("layer,width,rows", [
    (cases.general_delta(32, 64, 6144), 2048, 1000),                                                             # in three pieces
    (cases.parallel(cases.left(16, 4, 128, 128, 512, 64), cases.right(16, 64, 128, [0.95] * 16), 6144), 2048, 900),   # in two, beside two
    (cases.general_delta(16, 64, 3072), 1024, 1601),                                                             # in three
    (cases.general_delta(16, 64, 384), 1024, 1601),                                                              # whole
])
def test_down_projection_in_pieces(decoder, tmp_path, layer, width, rows):
    """A prompt in one pass, where pieces of the down projection's reduction fill idle CUs, against portions too short for that: streams behind
    each layer and scores.  Both sides' sums are fp32; what they round to bf16 may part by a step, as against the oracle."""
    cfg = cases.config(256, width, [layer, layer])
    cases.write_model(str(tmp_path), cfg, cases.weights(cfg))
    tokens = cases.tokens_of(cfg, rows)
    places = sorted({0, 63, 127, 128, rows // 2, rows - 2, rows - 1})
    whole = decoder.Decoder(str(tmp_path), rows, max_rows=rows)
    logits, streams = whole.step(whole.open(), tokens, places, streams=True)
    portions = decoder.Decoder(str(tmp_path), rows, max_rows=400)
    s, parts, scores = portions.open(), [], []
    for at in range(0, rows, 400):
        got, stream = portions.step(s, tokens[at:at + 400], [p - at for p in places if at <= p < at + 400], streams=True)
        parts.append(stream)
        scores.append(got)
    want = np.concatenate(parts, axis=1)
    for i in range(2):
        assert cases.error(streams[i], want[i]) < LIMIT[False], i
    assert cases.error(logits, np.concatenate(scores)) < LIMIT[False]


@pytest.mark.parametrize("layer,rows", [
    (cases.general_delta(16, 64, 3072), 300),                                                                    # three pieces
    (cases.parallel(cases.left(16, 4, 64, 64, 512, 64), cases.right(8, 64, 128, [0.95] * 8), 3072), 400),        # two, beside two; wide blocks in front
])
def test_linears_of_a_long_fp32_prompt(decoder, tmp_path, layer, rows):
    """A prompt in one pass, whose linears have their inputs split beforehand and the down projection in pieces, against portions of nine rows at most, which
    take the kernels of few rows: streams behind each layer and scores."""
    cfg = cases.config(256, 1024, [layer, layer])
    cases.write_model(str(tmp_path), cfg, cases.weights(cfg))
    tokens = cases.tokens_of(cfg, rows)
    places = sorted({0, 63, 64, 127, rows // 2, rows - 2, rows - 1})
    whole = decoder.Decoder(str(tmp_path), rows, float32=True, max_rows=rows)
    logits, streams = whole.step(whole.open(), tokens, places, streams=True)
    portions = decoder.Decoder(str(tmp_path), rows, float32=True, max_rows=9)
    s, parts, scores = portions.open(), [], []
    for at in range(0, rows, 9):
        got, stream = portions.step(s, tokens[at:at + 9], [p - at for p in places if at <= p < at + 9], streams=True)
        parts.append(stream)
        scores.append(got)
    want = np.concatenate(parts, axis=1)
    for i in range(2):
        assert cases.error(streams[i], want[i]) < LIMIT[True], i
    assert cases.error(logits, np.concatenate([x for x in scores if len(x)])) < LIMIT[True]


@pytest.mark.parametrize("width,ff,rows", [(1100, 3072, 200), (2100, 2048, 300)])
def test_norms_that_leave_their_rows_split(decoder, tmp_path, width, ff, rows):
    """A prompt whose feed-forward takes the second norm's rows as that left them, rows of two and of four vectors a thread with zeros behind them, against
    portions of nine rows, as above."""
    cfg = cases.sandwich(200, width, [cases.retention(4, 64, 64, [0.9, 0.99, 0.5, 0.0], cases.dense(ff))], (11, 6, 7))
    cases.write_model(str(tmp_path), cfg, cases.weights(cfg))
    tokens, places = cases.tokens_of(cfg, rows), [0, 63, 64, rows - 1]
    whole = decoder.Decoder(str(tmp_path), rows, float32=True, max_rows=rows)
    logits, streams = whole.step(whole.open(), tokens, places, streams=True)
    portions = decoder.Decoder(str(tmp_path), rows, float32=True, max_rows=9)
    s, parts, scores = portions.open(), [], []
    for at in range(0, rows, 9):
        got, stream = portions.step(s, tokens[at:at + 9], [p - at for p in places if at <= p < at + 9], streams=True)
        parts.append(stream)
        scores.append(got)
    assert cases.error(streams[0], np.concatenate(parts, axis=1)[0]) < LIMIT[True]
    assert cases.error(logits, np.concatenate([x for x in scores if len(x)])) < LIMIT[True]


@pytest.mark.parametrize("float32", [False, True])
def test_pieces_of_a_reduction_take_memory_only_where_one_is_cut(decoder, tmp_path, float32):
    """A narrow model's output linears are never cut, nor are its inputs split in the 32-bit mode: its feed-forward takes the rows of its channels more than
    the same model without, and no planes for sums (64 MiB here) or parts (144 MiB)."""
    import torch
    rows, used = 65536, []
    for i, ff in enumerate((None, None, 300)):                 # (the first loads the library's code as well)
        where = tmp_path / str(i)
        where.mkdir()
        cfg = cases.config(100, 128, [cases.parallel(cases.left(2, 1, 32, 32, 64, 32), cases.right(2, 16, 32, [0.9, 0.99]), ff)])
        cases.write_model(str(where), cfg, cases.weights(cfg))
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        engine = decoder.Decoder(str(where), rows, float32=float32, max_rows=rows)
        used.append(before - torch.cuda.mem_get_info()[0])
        engine.close_model()
    channels = rows * 384 * (4 if float32 else 2)              # 300 padded to 384
    assert used[2] - used[1] < channels + (16 << 20), used     # (allocations come in pieces of two MiB)


@pytest.mark.parametrize("rows", [1601, 1900])                   # in two; below 1537 rows whole
def test_a_layer_without_feed_forward_is_cut_in_front_of_its_norm(decoder, tmp_path, rows):
    """The last output linear of a parallel layer without feed-forward is the decayed attention's, whose sum is normed before it is added: its pieces come
    together first.  Between layers with one; against portions too short for a cut, as above."""
    mixers = cases.left(4, 2, 64, 64, 512, 64), cases.right(16, 64, 128, [0.95] * 16)
    cfg = cases.config(256, 1024, [cases.parallel(*mixers, 3072), cases.parallel(*mixers, None), cases.general_delta(16, 64, 3072)])
    cases.write_model(str(tmp_path), cfg, cases.weights(cfg))
    tokens = cases.tokens_of(cfg, rows)
    places = [0, 127, rows // 2, rows - 1]
    whole = decoder.Decoder(str(tmp_path), rows, max_rows=rows)
    logits, streams = whole.step(whole.open(), tokens, places, streams=True)
    portions = decoder.Decoder(str(tmp_path), rows, max_rows=400)
    s, parts, scores = portions.open(), [], []
    for at in range(0, rows, 400):
        got, stream = portions.step(s, tokens[at:at + 400], [p - at for p in places if at <= p < at + 400], streams=True)
        parts.append(stream)
        scores.append(got)
    want = np.concatenate(parts, axis=1)
    for i in range(3):
        assert cases.error(streams[i], want[i]) < LIMIT[False], i
    assert cases.error(logits, np.concatenate(scores)) < LIMIT[False]
