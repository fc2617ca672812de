"""Split records without a live token (m = -3e38, l = 0, acc = 0): a row of
such records alone combines to 0, and a row whose first record chunk holds only
such records to its other records, in the stand-alone combine, the fused
combine and the combine launch of wide GQA groups."""
import math

import numpy as np
import pytest

from gpu_helpers import dev, host
from oracle_bindings import bf16_to_f32, f32_to_bf16
from test_gpu_decode import build_cache, check_out

pytestmark = pytest.mark.gpu


def setup(oracle, seed, ctx, G, H, d, S=16):
    rng = np.random.default_rng(seed)
    P = sum((c + S - 1) // S for c in ctx) + 4
    kc, vc, sc, tables, signs, isl = build_cache(oracle, rng, ctx, H, d, S, P)
    q = f32_to_bf16(rng.standard_normal((len(ctx), G * H, d)).astype(np.float32))
    gate = rng.standard_normal(q.shape).astype(np.float32)
    return kc, vc, sc, tables, signs, float(isl), q, gate, P


@pytest.mark.parametrize("d,K", [(64, 1), (128, 4), (256, 8), (128, 16), (128, 33)])
@pytest.mark.parametrize("stage", [0, 1, 2])
def test_combine_of_an_empty_sequence(tq4, oracle, d, K, stage):
    G, H, S = 4, 2, 16
    ctx = [16 * K, 0, 5]
    kc, vc, sc, tables, signs, isl, q, gate, P = setup(oracle, d + K, ctx, G, H, d)
    rec = tq4.paged_decode_partials(dev(q), dev(kc), dev(vc), dev(sc), dev(tables),
                                    dev(np.array(ctx, np.int32)), dev(signs), H, S, P, K,
                                    inv_sqrt_len=isl)
    out = host(tq4.splitk_combine(rec, dev(signs), 3, G * H, d, K, gate=dev(gate),
                                  inv_sqrt_len=isl, output_stage=stage))
    assert np.all(np.isfinite(bf16_to_f32(out)))
    assert not np.any(bf16_to_f32(out)[1])


# one launch (G = 4), two launches (G = 16; d = 256, G = 8, K = 8), the
# persistent kernel (B = 160), one live split
@pytest.mark.parametrize("B,G,d,K", [(3, 4, 64, 2), (3, 4, 128, 4), (3, 4, 256, 20), (3, 16, 64, 3),
                                     (3, 16, 128, 4), (3, 16, 128, 33), (3, 8, 256, 8),
                                     (160, 3, 128, 8), (3, 4, 128, 1)])
def test_fused_without_a_valid_page(tq4, oracle, B, G, d, K):
    H, S = (4 if B > 3 else 2), 16
    ctx = [16 * K] * B
    ctx[-1] = 16 * K - 3
    kc, vc, sc, tables, signs, isl, q, gate, P = setup(oracle, B + G + d + K, ctx, G, H, d)
    bad = tables.copy()
    bad[1] = -1
    bad[-1] = P + 5
    ws = tq4.decode_workspace(B, G * H, H, d, K)
    for _ in range(2):  # the workspace is left as it was found
        out = host(tq4.paged_decode(dev(q), dev(kc), dev(vc), dev(sc), dev(bad),
                                    dev(np.array(ctx, np.int32)), dev(signs), H, S, P,
                                    workspace=ws, gate=dev(gate), num_splits=K,
                                    inv_sqrt_len=isl, output_stage=2))
        assert np.all(np.isfinite(bf16_to_f32(out)))
        assert not np.any(bf16_to_f32(out)[[1, -1]])
        assert np.any(bf16_to_f32(out)[0])
    assert tq4.decode_poll_timeouts(ws, B, H) == 0


@pytest.mark.parametrize("G,d", [(4, 128), (16, 128), (8, 256)])
@pytest.mark.parametrize("entry", ["fused", "combine"])
def test_neutral_first_chunk(tq4, oracle, G, d, entry):
    """32 splits of one page, the first 16 (a whole record chunk) invalid."""
    H, S, K = 2, 16, 32
    ctx = [S * K]
    kc, vc, sc, tables, signs, isl, q, _, P = setup(oracle, 5 * G + d, ctx, G, H, d)
    bad = tables.copy()
    bad[0, :16] = -1
    scale = np.float32(1.0 / math.sqrt(d))
    _, want = oracle.paged_decode(q, kc, vc, sc, np.ascontiguousarray(tables[:, 16:]),
                                  np.array([S * 16], np.int32), signs, None, G * H, H, d, S, P, 16,
                                  scale, np.float32(isl), 1, threads=8)
    args = [dev(q), dev(kc), dev(vc), dev(sc), dev(bad), dev(np.array(ctx, np.int32)), dev(signs),
            H, S, P]
    if entry == "fused":
        out = tq4.paged_decode(*args, num_splits=K, inv_sqrt_len=isl)
    else:
        rec = tq4.paged_decode_partials(*args, K, inv_sqrt_len=isl)
        out = tq4.splitk_combine(rec, dev(signs), 1, G * H, d, K, inv_sqrt_len=isl)
    check_out(host(out), want, f"neutral first chunk G {G} d {d} {entry}")


def test_nan_record_stays_nan(tq4):
    """A record that holds NaN (here its m) is not taken for a neutral one."""
    import torch
    d, K = 128, 4
    rec = torch.zeros((1, 2, K, d + 4), device="cuda")
    rec[..., 1] = 1.0
    rec[0, 1, 2, 0] = float("nan")
    out = tq4.splitk_combine(rec, None, 1, 2, d, K, output_stage=0).float()
    assert not torch.any(out[0, 0]) and torch.all(torch.isnan(out[0, 1]))
