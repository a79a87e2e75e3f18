"""Which attention a batch of one conversation takes (host logic: no GPU): the sides on which measured launches were the faster ones."""
import pytest

F16, Q8_0 = 1, 8
L8, L7, MID, SMALL, TEXT = (Q8_0, 32, 8, 128), (F16, 32, 32, 128), (F16, 32, 16, 64), (F16, 32, 4, 64), (F16, 12, 12, 64)


@pytest.fixture(scope="module")
def takes(pkg):
    lib = pkg.load_library()
    return lambda model, n, past, encoder=0: int(lib.mi355_debug_attn_plan(*model, n, past + n, encoder)) > 0


@pytest.mark.parametrize("model,yes,no", [
    (L8, [(2, 2100), (3, 1900), (5, 1495), (14, 700), (31, 200), (40, 0), (37, 160), (64, 613)], [(2, 700), (5, 900), (8, 700), (12, 400), (22, 200), (31, 150), (32, 0), (1, 3900)]),
    (L7, [(2, 3000), (3, 1900), (5, 900), (12, 400), (32, 0)], [(2, 2100), (14, 200)]),
    (MID, [(3, 1900), (8, 700), (22, 200)], [(14, 200), (2, 700)]),
    (SMALL, [(2, 0), (3, 0), (31, 20), (3, 1900), (8, 700), (22, 200), (14, 200), (2, 700)], []),                  # fewer than 1024 values of K a row: no one-token kernel beside the columns
    ((Q8_0, 28, 4, 128), [(2, 0), (2, 60), (8, 500), (31, 30)], []),
])
def test_short_batches(takes, model, yes, no):
    assert [c for c in yes if not takes(model, *c)] == [] and [c for c in no if takes(model, *c)] == []


@pytest.mark.parametrize("model,yes,no", [
    (L8, [(256, 3500), (450, 3400), (512, 0), (512, 700), (512, 1400)], [(512, 2488), (512, 3400), (513, 0)]),
    (L7, [(256, 3500), (300, 2000), (512, 0), (512, 1000)], [(400, 2500), (450, 1500), (512, 1500), (512, 2500)]),
    (SMALL, [(256, 0), (700, 900), (768, 1200)], [(850, 0), (1024, 900)]),
])
def test_long_batches(takes, model, yes, no):
    assert [c for c in yes if not takes(model, *c)] == [] and [c for c in no if takes(model, *c)] == []


def test_texts(takes):
    assert all(takes(TEXT, n, 0, 1) for n in (3, 20, 187, 700, 2000, 2048))


@pytest.mark.parametrize("model,n,bytes_", [
    (L8, 225, 4096 * 8 * 128 * 4), (L7, 897, 4096 * 32 * 128 * 2), ((Q8_0, 16, 8, 128), 449, 4096 * 8 * 128 * 4), (SMALL, 225, 4096 * 4 * 64 * 2), ((Q8_0, 56, 8, 128), 225, 4096 * 8 * 128 * 4)])
def test_planes_workspace(pkg, model, n, bytes_):
    """A context keeps the V planes' workspace from the first micro-batch of eight query tiles (of 128, 64, 32 tokens with 1, 2, more query heads to a kv head) on, and not below."""
    plan = pkg.load_library().mi355_debug_attn_planes_plan
    assert [plan(*model, 4096, t) for t in (1, 32, n - 1)] == [0] * 3
    assert [plan(*model, 4096, t) for t in (n, 2048)] == [bytes_] * 2


@pytest.mark.parametrize("model", [(Q8_0, 12, 4, 64), (F16, 28, 4, 64), (F16, 10, 2, 64), (2, 32, 8, 128), (Q8_0, 32, 2, 128), (Q8_0, 32, 8, 96)])
def test_no_planes_workspace_without_a_form(pkg, model):
    """64-wide heads in threes, fives, sixes, sevens; a q4_0 cache; more than eight query heads to a kv head; other widths."""
    assert pkg.load_library().mi355_debug_attn_planes_plan(*model, 4096, 2048) == 0


@pytest.mark.parametrize("model,yes,no", [
    (L8, [(850, 0), (520, 300), (1024, 0), (1919, 2048), (300, 2000)], [(520, 0), (600, 0), (700, 0), (224, 3500)]),
    ((F16, 64, 8, 128), [(850, 0), (600, 300), (1024, 0)], [(260, 0), (520, 0), (700, 0)]),
    ((Q8_0, 40, 8, 128), [(700, 0), (520, 300)], [(420, 0), (520, 0)]),
    (L7, [(1000, 0), (2000, 2000)], [(896, 3000)]),
    (SMALL, [(850, 300), (800, 1100), (2000, 1000), (1024, 1000)], [(1024, 0), (1600, 0), (2000, 0), (1600, 500)]),
    ((F16, 64, 8, 64), [(2000, 0), (1600, 500)], [(520, 0), (950, 0)]),
])
def test_planes_where_they_pay(pkg, model, yes, no):
    """Launches timed with and without the V planes of a prompt's attention, the planes' own launch among them: fresh prompts of few keys convert for themselves."""
    taken = pkg.load_library().mi355_debug_attn_planes_taken
    assert [c for c in yes if taken(*model, c[0], sum(c), sum(c)) != 1] == [] and [c for c in no if taken(*model, c[0], sum(c), sum(c)) != 0] == []


def test_planes_of_several_conversations(pkg):
    """Four prompts of 500 tokens in one batch: a query sees 250 keys of 2000 on average, as many as in the prompt alone, for four times the tiles; sixteen of 125 see too few for the cells scanned."""
    taken = pkg.load_library().mi355_debug_attn_planes_taken
    assert taken(*L8, 2000, 2000, 500) == 1 and taken(*L8, 2000, 2000, 125) == 0
