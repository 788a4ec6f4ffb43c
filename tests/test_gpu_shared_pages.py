"""Decode steps whose rows share pages (forked sequences): the pages attended once for a tile of rows and merged with each row's
own, against the same rows decoded one at a time."""
import numpy as np
import pytest

from retrograd_amd import engine as E
from retrograd_amd import synth

pytestmark = pytest.mark.gpu

# head width and query heads over 8 kv heads: tiles of 128, 64, 40, 32, 24 rows
HEADS = {"128x1": (128, 8), "64x2": (64, 16), "64x3": (64, 24), "128x4": (128, 32), "64x5": (64, 40)}


@pytest.mark.parametrize("heads", list(HEADS))
def test_shared_pages_match_rows_decoded_alone(tmp_path, heads):
    """A prefix of 32 pages and a bit, six prompts of 0 to 300 tokens over it, each forked into up to 50 rows with 1 to 70 tokens
    of their own; among them rows that share nothing, one whose first positions are gone, and lengths on both sides of a page's
    end. One layer; queries and probabilities carry 22 bits and sums are f32, which leaves about 1e-6 of the logits: 1e-5 is
    asked of nine rows in ten. A row's new key and value come from products over another number of tokens, so they may sit on the
    other side of a rounding boundary of the cache: no row is further off than one such step (2^-11 of a value) in one dimension of a
    head whose whole weight lies on that token."""
    dim, n_head = HEADS[heads]
    shape = synth.scaled(synth.TINY_LLAMA, n_layer=1, n_embd=512, n_head=n_head, n_head_kv=8, head_dim=dim, n_ff=512, name="shared-%s" % heads)
    path = tmp_path / "m.gguf"
    synth.write_model(path, shape, seed=5, device="cpu", std=0.08)
    rng = np.random.default_rng(6)
    tokens = lambda n: rng.integers(0, shape.n_vocab, n).astype(np.int32)
    with E.Engine(path, E.EngineConfig(n_ctx=65536, n_seq_max=256, n_batch=2048, n_ubatch=2048)) as eng:
        end, slot = {}, 0
        eng.step_logits([(0, tokens(1042), 0)], [])
        for prompt in (0, 14, 78, 300, 33, 1):
            first = slot
            if first:
                eng.seq_cp(0, first, 0, 1042)
            if prompt:
                eng.step_logits([(first, tokens(prompt), 1042)], [])
            for k in range(40 if prompt != 14 else 13):
                if slot != first:
                    eng.seq_cp(first, slot, 0, 1042 + prompt)
                end[slot] = 1042 + prompt
                slot += 1
        for lone in range(20):                   # nothing in common with anyone, between the others' tiles when rows are shuffled
            eng.step_logits([(slot, tokens(1 + 40 * (lone % 3)), 0)], [])
            end[slot] = 1 + 40 * (lone % 3)
            slot += 1
        forks = [s for s in end if s < 213 and s % 5 == 1]
        for s in forks:                          # what a row has of its own
            own = 1 + (s * 7) % 70
            eng.step_logits([(s, tokens(own), end[s])], [])
            end[s] += own
        eng.seq_rm(214, 0, 20)
        order = list(end)
        new = {s: tokens(1) for s in order}
        alone = []
        for s in order:
            alone.append(eng.step_logits([(s, new[s], end[s])], [(0, 0)])[0])
            eng.seq_rm(s, end[s], end[s] + 1)
        for rows in (order, [order[i] for i in rng.permutation(len(order))]):
            eng.profile(2)
            got = eng.step_logits([(s, new[s], end[s]) for s in rows], [(r, 0) for r in range(len(rows))])
            launches = eng.profile_read()["rope"][1]
            eng.profile(0)
            for s in rows:
                eng.seq_rm(s, end[s], end[s] + 1)
            want = np.stack([alone[order.index(s)] for s in rows])
            assert np.isfinite(got).all()
            worst = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
            print("%s: rotation launches %d, nine of ten %.2e, worst row %.2e" % (heads, launches, np.quantile(worst, 0.9), worst.max()), flush=True)
            assert rows is not order or launches == 1          # (in order the shared pages are worth their launches)
            assert np.quantile(worst, 0.9) <= 1e-5
            assert worst.max() <= 2.0 ** -11 / np.sqrt(dim / 3)
