"""reshape_scatter over requests of several tokens (cu_seqlens): the device
takes a request in 16-token chunks, the oracle walks its tokens in order. Every
byte of the pool must agree, for prompts that begin anywhere in a strip and for
slots in any order, strips that several chunks touch and slots written twice
(the later token wins)."""
import numpy as np
import pytest

from oracle_bindings import f32_to_bf16
from test_gpu_scatter import assert_same, scatter_pair

pytestmark = pytest.mark.gpu


def positions(rng, pages, S, begin, n):
    """The slots of positions begin .. begin + n - 1 over the given pages."""
    at = np.arange(begin, begin + n)
    return pages[at // S] * S + at % S


def layout(kind, rng, pages, S, n):
    """n slots inside the request's own pages."""
    cap = len(pages) * S
    s = positions(rng, pages, S, int(rng.integers(0, cap - n + 1)), n)
    if kind == "shuffled":
        s = rng.permutation(s)
    elif kind == "interleaved":  # two strips in turn: every chunk touches both
        s = np.where(np.arange(n) % 2 == 0, s[0] // 16 * 16, s[-1] // 16 * 16) + \
            (np.arange(n) // 2) % 16
    elif kind == "rewritten":  # later tokens write earlier tokens' slots again
        s[n // 2:] = s[rng.integers(0, max(1, n // 2), n - n // 2)]
    elif kind == "reversed":
        s = s[::-1].copy()
    elif kind == "pads":
        s[rng.random(n) < 0.3] = -1
    return s


def case(tq4, oracle, rng, lens, kinds, H, d, S, scale=1.0, **kw):
    R = len(lens)
    need = [n // S + 2 for n in lens]
    P = sum(need) + 2
    perm, at, slots = rng.permutation(P), 0, []
    for n, m, kind in zip(lens, need, kinds):
        if n:
            slots.append(layout(kind, rng, perm[at:at + m], S, n))
        at += m
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    x = rng.standard_normal((2, T, H, d)) * scale
    key, val = (f32_to_bf16(x[i].astype(np.float32)) for i in range(2))
    nb = P * H * S * d // 2
    prior = (rng.integers(-128, 128, nb, dtype=np.int8), rng.integers(-128, 128, nb, dtype=np.int8),
             rng.standard_normal(2 * P * H * S).astype(np.float32))
    sl = np.concatenate(slots).astype(np.int32)
    got, want = scatter_pair(tq4, oracle, key, val, sl, cu, R, H, d, S, P, prior=prior, **kw)
    assert_same(got, want)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("S", [16, 64])
def test_prompts_at_tile_edges(tq4, oracle, d, S):
    """Lengths around one and several chunks, begun at random places, empty
    requests among them, and a head count that no group size divides."""
    rng = np.random.default_rng(d + S)
    lens = [1, 15, 16, 17, 0, 31, 32, 33, 2, 48, 0, 130]
    case(tq4, oracle, rng, lens, ["prompt"] * len(lens), 3, d, S)


@pytest.mark.parametrize("kind", ["shuffled", "interleaved", "rewritten", "reversed", "pads"])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_any_slot_order(tq4, oracle, kind, d):
    rng = np.random.default_rng(d)
    lens = [1, 2, 16, 37, 64, 90]
    case(tq4, oracle, rng, lens, [kind] * len(lens), 5, d, 32)


def test_long_prompt_takes_heads_together(tq4, oracle):
    """More (chunk, head) pairs than the launch offers workgroups: several
    heads, then whole chunks, to a workgroup; a rewritten tail in the last."""
    rng = np.random.default_rng(77)
    case(tq4, oracle, rng, [5003], ["prompt"], 8, 128, 16)
    case(tq4, oracle, rng, [17000], ["prompt"], 2, 64, 128)
    case(tq4, oracle, rng, [2100], ["rewritten"], 8, 64, 16)


def test_many_requests_and_item_windows(tq4, oracle):
    """More requests than workgroups offered, and item windows that begin and
    end inside a request's heads."""
    rng = np.random.default_rng(78)
    lens = [int(x) for x in rng.integers(0, 4, 2500)]
    case(tq4, oracle, rng, lens, ["prompt"] * 2500, 1, 64, 16)
    lens = [20, 3, 0, 41, 16]
    for begin, count in ((0, 1), (2, 5), (3, 12), (7, 13), (19, 1), (6, 100)):
        case(tq4, oracle, rng, lens, ["prompt"] * 5, 4, 128, 32, item_begin=begin,
             item_count=count)


@pytest.mark.parametrize("d", [64, 256])
def test_extreme_rows(tq4, oracle, d):
    """Rows whose scale has no normal power of two (absmax down to the smallest
    BF16 numbers), all-zero rows and large ones, in full and partial chunks."""
    rng = np.random.default_rng(79)
    lens = [16, 23, 64]
    scale = np.exp2(rng.integers(-132, 120, (sum(lens), 1, 1)).astype(np.float64))
    scale[::7] = 0.0
    case(tq4, oracle, rng, lens, ["prompt"] * 3, 2, d, 16, scale=scale)


@pytest.mark.parametrize("R", [1, 3, 1023, 1024, 1025, 2050])
@pytest.mark.parametrize("H", [1, 3])
def test_request_counts_around_the_staged_plan(tq4, oracle, R, H):
    """Request counts at the edges of the on-chip plan (1024 requests, four a
    thread), empty ones and short and longer ones among them."""
    rng = np.random.default_rng(80 + R + H)
    lens = [int(x) for x in rng.choice([0, 1, 1, 2, 5, 16, 17, 40], R)]
    lens[-1] = 19
    case(tq4, oracle, rng, lens, ["prompt"] * R, H, 64, 16)


@pytest.mark.parametrize("kind,n", [("prompt", 270001), ("rewritten", 40000), ("pads", 40000)])
def test_more_chunks_than_a_group(tq4, oracle, kind, n):
    """Requests of more chunks than the workgroups check together (16 each, 1024
    workgroups), regular and with strips that far chunks share."""
    case(tq4, oracle, np.random.default_rng(n), [n, 7], [kind, "prompt"], 1, 64, 16)


@pytest.mark.parametrize("tail", ["plain", "shared", "swapped"])
def test_strips_of_one_table_place(tq4, oracle, tail):
    """The strips of a group's chunks all at one place of the strip table (equal
    modulo 256), a chunk that touches another's strip again, two chunks with
    their strips' halves swapped."""
    rng = np.random.default_rng(81)
    H, d, S, chunks = 2, 64, 16, 40
    P = 256 * chunks
    strips = 256 * rng.permutation(chunks) + 5
    slots = (strips[:, None] * 16 + np.arange(16)).reshape(-1)
    if tail == "shared":
        slots[-16:] = slots[48:64]
    elif tail == "swapped":
        slots[32:40], slots[320:328] = slots[320:328].copy(), slots[32:40].copy()
    T = len(slots)
    key, val = (f32_to_bf16(rng.standard_normal((T, H, d)).astype(np.float32)) for _ in range(2))
    nb = P * H * S * d // 2
    prior = (rng.integers(-128, 128, nb, dtype=np.int8), rng.integers(-128, 128, nb, dtype=np.int8),
             rng.standard_normal(2 * P * H * S).astype(np.float32))
    got, want = scatter_pair(tq4, oracle, key, val, slots.astype(np.int32),
                             np.array([0, T], np.int32), 1, H, d, S, P, prior=prior)
    assert_same(got, want)
