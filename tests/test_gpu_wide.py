"""The sliced path (FP32 and bf16 rows spread over the chip) against the
float64 oracle: ids, consumption flags, statuses and kept sets exactly, float64
probabilities within 1e-12 relative.

Vocabulary sizes sit at the edges of the 8,192-token slices and of the 16- and
4-token vectors; rows are odd, strided, masked, penalised and biased."""
import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from deepseekrpc_amd import batch, workloads
from oracle import pcg64_oracle as P
from oracle import sampling_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def device_logits(x, dtype, pad=0):
    """``x`` (exact values of ``dtype``) on the device, rows ``pad`` elements apart beyond the vocabulary."""
    rows, V = x.shape
    t = torch.zeros(rows, V + pad, dtype=torch.float32)
    t[:, :V] = torch.from_numpy(x.astype(np.float32))
    return t.to(dtype).to(DEV)[:, :V]


def rows_of(rng, rows, V, kind, dtype):
    if kind == "flat":
        x = rng.uniform(-1e-3, 1e-3, (rows, V))
    elif kind == "normal":
        x = rng.normal(0, 3, (rows, V))
    else:
        x = rng.normal(0, 1, (rows, V))
        for r in range(rows):
            x[r, rng.choice(V, 24, replace=False)] += rng.uniform(6, 12, 24)
    x = x.astype(np.float32)
    return workloads.bf16_round(x) if dtype == torch.bfloat16 else x


def sample(x, pols, u, dtype, pad=0, counts=None, gens=None, biases=None, allowed=None, **kw):
    V = x.shape[1]
    hist = None if counts is None else batch.HistoryTable.from_dense(counts, gens, device=DEV)
    bias = None if biases is None else batch.BiasTable.from_dicts(biases, device=DEV)
    allow = None if allowed is None else torch.from_numpy(batch.pack_allow(allowed).view(np.int32)).to(DEV)
    res = batch.sample_rows(device_logits(x, dtype, pad), pols, history=hist, bias=bias, allow_bits=allow,
                            uniforms=torch.from_numpy(np.asarray(u)).to(DEV), probs="f64", kept=True, **kw)
    torch.cuda.synchronize()
    kept = batch.unpack_bits(res.kept_bits.cpu().numpy().view(np.uint32), V)
    probs = res.probs.cpu().numpy()
    flags = res.flags.cpu().numpy()
    for r in range(len(pols)):
        ref = O.sample_row(x[r], O.Policy(**pols[r]), float(u[r]), None if counts is None else counts[r],
                           None if gens is None else gens[r], None if biases is None else biases[r],
                           None if allowed is None else allowed[r])
        assert int(res.status[r]) == ref.status, (r, int(res.status[r]), ref.status, pols[r])
        if ref.status:
            continue
        got = (int(res.tokens[r]), bool(res.consumed[r]))
        assert got == (ref.token, ref.consumed), (r, got, ref.token, ref.margin, pols[r], hex(int(flags[r])))
        np.testing.assert_array_equal(kept[r], ref.topk_kept, err_msg=f"row {r} {pols[r]}")
        np.testing.assert_allclose(probs[r], ref.probs, rtol=1e-12, atol=1e-300, err_msg=f"row {r} {pols[r]}")
    return flags


WHOLE = [dict(top_p=0.9), dict(temperature=0.7, top_p=0.95), dict(min_p=0.05), dict(temperature=1.3, top_p=0.8, min_p=0.02),
         dict(top_p=0.0), dict(min_p=1.0), dict(top_p=0.999, min_p=1e-4), dict(temperature=0.0), dict(temperature=0.3, top_p=0.5)]
TOPK = [dict(temperature=0.7, top_k=50, top_p=0.9), dict(top_k=1), dict(top_k=1024, top_p=0.99), dict(temperature=0.0),
        dict(temperature=1.4, top_k=300, min_p=0.01), dict(top_k=17)]
PEN = dict(repetition_penalty=1.2, presence_penalty=0.4, frequency_penalty=0.2)


def histories(rng, rows, V, longest):
    counts = np.zeros((rows, V), np.int32)
    gens = np.zeros((rows, V), np.int32)
    for r in range(rows):
        h = rng.integers(0, V, int(rng.integers(1, longest)))
        counts[r] = np.bincount(h, minlength=V)
        gens[r] = np.minimum(counts[r], np.bincount(h[len(h) // 3:], minlength=V))
    return counts, gens


# One slice, a slice and one token, vectors cut short, the largest.
SIZES = [8192, 8193, 16384, 16399, 24575, 129280]


@pytest.mark.parametrize("V", SIZES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("family", ["whole", "topk", "mixed"])
def test_penalised_and_biased_rows(V, dtype, family):
    rng = np.random.default_rng(V + 7 * (dtype == torch.bfloat16))
    pols = {"whole": WHOLE, "topk": TOPK, "mixed": WHOLE + TOPK}[family]
    pols = [dict(p, **(PEN if r % 4 else dict(repetition_penalty=0.8, presence_penalty=-0.3))) for r, p in enumerate(pols)]
    B = len(pols)
    x = np.concatenate([rows_of(rng, 1, V, ("spiked", "normal")[r % 2], dtype) for r in range(B)])
    counts, gens = histories(rng, B, V, min(6000, V // 5))
    biases = [{int(t): float(rng.uniform(-8, 8)) for t in rng.choice(V, int(rng.integers(1, 60)), replace=False)}
              for _ in range(B)]
    biases[1] = {}
    allowed = rng.random((B, V)) < 0.9
    u = rng.random(B)
    flags = sample(x, pols, u, dtype, 3, counts, gens, biases, allowed)
    # A row with fewer 16-token groups than its top-k may go to the general path; so do short rows of batches that
    # are not all top-k or greedy, for which that path is the faster one.
    on = np.array([p.get("top_k", 0) <= V // 16 and (V >= 16384 or family == "topk") for p in pols])
    assert (flags & N.FLAG_SPLIT).astype(bool)[on].all(), [hex(int(f)) for f in flags]


@pytest.mark.parametrize("V", SIZES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_without_tables(V, dtype):
    """No history or bias; odd strides and sizes keep bf16 rows off the register kernels."""
    rng = np.random.default_rng(V + 77)
    pols = WHOLE + TOPK + [dict(), dict(temperature=1.7)]
    B = len(pols)
    x = np.concatenate([rows_of(rng, 1, V, ("spiked", "normal", "flat")[r % 3], dtype) for r in range(B)])
    u = rng.random(B)
    sample(x, pols, u, dtype, 5)
    sample(x, pols, u, dtype, 5, allowed=rng.random((B, V)) < 0.5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_flat_and_tied_rows(dtype):
    """Ties at the top-p and top-k cuts, cut by index, and rows the path hands over."""
    rng = np.random.default_rng(99)
    V = 20000
    pols = [dict(top_p=0.9, **PEN), dict(top_p=0.37, **PEN), dict(top_p=0.5, min_p=0.5, **PEN), dict(top_k=700, top_p=0.6, **PEN),
            dict(top_k=64, **PEN), dict(top_p=0.61, temperature=0.2, **PEN), dict(top_p=0.999999, **PEN), dict(**PEN)]
    B = len(pols)
    grid = workloads.bf16_round((np.round(rng.normal(0, 1, (B, V)) * 8) / 8).astype(np.float32))
    flat = rows_of(rng, B, V, "flat", dtype)
    equal = np.full((B, V), 0.25, np.float32)
    counts, gens = histories(rng, B, V, 3000)
    u = rng.random(B)
    for x in (grid, flat, equal):
        sample(x, pols, u, dtype, 1, counts, gens)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_invalid_rows_report_in_order(dtype):
    V, B = 9000, 7
    rng = np.random.default_rng(5)
    x = rows_of(rng, B, V, "spiked", dtype)
    x[0, 8999] = np.nan
    x[1, 17] = np.inf
    x[2, 8191] = -np.inf   # masked, not invalid
    allowed = np.ones((B, V), bool)
    allowed[3] = False
    allowed[1, 17] = False  # a masked +inf still counts
    allowed[4, :] = False
    allowed[4, 8999] = True
    pols = [dict(top_p=0.9), dict(top_k=5), dict(top_k=5), dict(top_p=0.9), dict(min_p=0.1), dict(top_k=3),
            dict(top_p=0.9, temperature=0.5)]
    u = rng.random(B)
    u[6] = 1.0
    sample(x, pols, u, dtype, 1, allowed=allowed)


def test_invalid_tables_take_the_general_path():
    V = 20000
    rng = np.random.default_rng(6)
    x = rows_of(rng, 6, V, "spiked", torch.float32)
    d = DEV
    # Ids out of order across slices, inside one slice, out of range, counts above the limit, generated above counts; row 5 valid.
    ids = [[9000, 5], [7, 7], [5, V], [3, 9], [4], [5, 9000]]
    cnt = [[1, 1], [1, 1], [1, 1], [600_000, 600_000], [1], [2, 1]]
    gen = [[1, 1], [1, 1], [1, 1], [0, 0], [2], [1, 1]]
    off = np.concatenate([[0], np.cumsum([len(i) for i in ids])])
    t = lambda a: torch.tensor(np.concatenate(a), dtype=torch.int32, device=d)
    h = batch.HistoryTable(torch.tensor(off, device=d), t(ids), t(cnt), t(gen))
    for pol in (dict(top_p=0.9, **PEN), dict(top_k=9, **PEN)):
        res = batch.sample_rows(device_logits(x, torch.float32, 1), [pol] * 6, history=h,
                                uniforms=torch.full((6,), 0.4, dtype=torch.float64, device=d))
        torch.cuda.synchronize()
        assert res.status.cpu().tolist() == [N.E_COUNTS] * 4 + [N.E_GENERATED, 0]
        flags = res.flags.cpu().numpy()
        assert ((flags[:5] >> 4) == 6).all() and flags[5] & N.FLAG_SPLIT


def test_device_draws_and_single_tokens():
    rng = np.random.default_rng(8)
    B, V = 6, 33001
    x = rows_of(rng, B, V, "spiked", torch.float32)
    pols = [dict(top_p=0.9, **PEN), dict(top_k=40, **PEN), dict(top_p=0.0, **PEN), dict(temperature=0.0, **PEN), dict(min_p=0.3, **PEN),
            dict(temperature=0.01, **PEN)]
    counts, gens = histories(rng, B, V, 500)
    gensr = [np.random.default_rng(70 + r) for r in range(B)]
    st0 = [g.bit_generator.state["state"] for g in gensr]
    states = batch.pcg64_states(gensr, DEV)
    res = batch.sample_rows(device_logits(x, torch.float32, 0), pols, rng_state=states,
                            history=batch.HistoryTable.from_dense(counts, gens, device=DEV))
    words = states.cpu().numpy().view(np.uint64)
    for r in range(B):
        nxt, u = P.random(st0[r]["state"], st0[r]["inc"])
        ref = O.sample_row(x[r], O.Policy(**pols[r]), u, counts[r], gens[r])
        assert (int(res.tokens[r]), bool(res.consumed[r])) == (ref.token, ref.consumed), r
        assert int(words[r, 0]) | (int(words[r, 1]) << 64) == (nxt if ref.consumed else st0[r]["state"]), r
