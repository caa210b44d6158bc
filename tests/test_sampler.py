"""GPU sampler (csrc/sampler.hip) vs the oracle restatement of
acorninfer/sampler.py:38-68: processed logits identical (kept set and
values), the drawn token identical to the oracle's inverse-CDF draw for the
same uniform, logprob within fp32 rounding; greedy rows; NaN/inf rows;
determinism and graph replay."""
import pytest
import torch

from oracle.sampler_ref import draw_ref, process_ref

CASES = [(0.7, 20, 0.95), (1.0, 0, 0.9), (0.6, 50, 1.0), (1.3, 0, 0.5), (1.0, 1, 1.0),
         (0.9, 0, 1.0), (0.8, 1000, 0.7), (1.0, 0, 0.999)]


def _rows(n, V, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(n, V, generator=g) * 3).to(dtype)


def _gpu(logits, params, us, processed=True):
    from acorninfer_amd.sampler import sample_batch
    B, V = logits.shape
    t = torch.tensor([p[0] for p in params], dtype=torch.float32, device="cuda")
    k = torch.tensor([p[1] for p in params], dtype=torch.int32, device="cuda")
    p_ = torch.tensor([p[2] for p in params], dtype=torch.float32, device="cuda")
    u = torch.tensor(us, dtype=torch.float32, device="cuda")
    proc = torch.empty(B, V, device="cuda") if processed else None
    tok, lp, st = sample_batch(logits.cuda(), t, k, p_, u, processed=proc)
    return tok.cpu(), lp.cpu(), st.cpu(), (proc.cpu() if processed else None)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_processed_and_draw_match_oracle(dtype):
    V = 151936
    logits = _rows(len(CASES), V, dtype, 11)
    us = [0.0, 0.37, 0.5, 0.91, 0.2, 0.999, 0.63, 0.05]
    tok, lp, st, proc = _gpu(logits, CASES, us)
    assert st.eq(0).all()
    for r, (t, k, p) in enumerate(CASES):
        want = process_ref(logits[r], t, k, p)
        kept_w, kept_g = want.isfinite(), proc[r].isfinite()
        if p > 0.99 and k == 0:
            # boundary inside the dense tail: HF's fp32 cumsum over ~1.5e5 tiny
            # probabilities decides elements within its own rounding; the
            # kernel sums exactly. Bound the mass of any disagreement.
            pr = torch.softmax((logits[r].float() / t).double(), 0)
            assert pr[kept_w ^ kept_g].sum() < 1e-5
            kept = kept_g
            torch.testing.assert_close(proc[r][kept], (logits[r].float() / t)[kept], rtol=0, atol=0)
            wt, wlp = draw_ref(proc[r], us[r])
        else:
            assert torch.equal(kept_w, kept_g), \
                f"row {r}: kept sets differ ({int(kept_w.sum())} vs {int(kept_g.sum())})"
            torch.testing.assert_close(proc[r][kept_g], want[kept_w], rtol=0, atol=0)
            wt, wlp = draw_ref(want, us[r])
        assert int(tok[r]) == wt, f"row {r}: token {int(tok[r])} vs {wt}"
        assert abs(float(lp[r]) - wlp) < 1e-4


@pytest.mark.gpu
def test_known_answers_and_greedy():
    logits = torch.tensor([[2.0, 1.0, 0.5, -1.0]] * 4)
    params = [(1.0, 1, 1.0), (1.0, 2, 1.0), (1.0, 0, 0.6), (0.0, 0, 1.0)]
    tok, lp, st, proc = _gpu(logits, params, [0.5, 0.99, 0.3, 0.7])
    assert tok.tolist()[0] == 0 and abs(float(lp[0])) < 1e-6
    assert proc[1][:2].isfinite().all() and proc[1][2:].isinf().all()
    assert proc[2][0].isfinite() and proc[2][1:].isinf().all() and int(tok[2]) == 0
    assert int(tok[3]) == 0 and float(lp[3]) == 0.0          # temperature 0: greedy


@pytest.mark.gpu
def test_nonfinite_rows_flagged_and_sampler_raises():
    from acorninfer_amd.sampler import Sampler, SamplingParams
    logits = torch.tensor([[1.0, float("nan"), 0.0], [1.0, 2.0, 0.0]])
    _, _, st, _ = _gpu(logits, [(1.0, 0, 1.0)] * 2, [0.5, 0.5], processed=False)
    assert st.tolist() == [1, 0]
    with pytest.raises(ValueError, match="NaN/inf"):
        Sampler(SamplingParams()).process(torch.tensor([1.0, float("inf")], device="cuda"))
    with pytest.raises(ValueError):
        Sampler(SamplingParams(temperature=0.0))


@pytest.mark.gpu
def test_sampler_class_matches_reference_api():
    from acorninfer_amd.sampler import Sampler, SamplingParams
    logits = _rows(1, 151936, torch.float32, 5)[0].cuda()
    s = Sampler(SamplingParams(temperature=0.7, top_k=20, top_p=0.95))
    torch.testing.assert_close(s.process(logits).cpu(), process_ref(logits.cpu(), 0.7, 20, 0.95),
                               rtol=0, atol=0)
    g1 = torch.Generator(device="cuda").manual_seed(42)
    g2 = torch.Generator(device="cuda").manual_seed(42)
    a = [Sampler(SamplingParams(), g1).sample(logits) for _ in range(5)]
    b = [Sampler(SamplingParams(), g2).sample(logits) for _ in range(5)]
    assert a == b


@pytest.mark.gpu
def test_empirical_frequencies_follow_processed_distribution():
    """Many uniforms on one small row: token frequencies match softmax(processed)."""
    V, n = 64, 4096
    logits = _rows(1, V, torch.float32, 9).repeat(n, 1)
    us = torch.rand(n, generator=torch.Generator().manual_seed(3)).tolist()
    tok, _, _, _ = _gpu(logits, [(0.8, 10, 0.9)] * n, us, processed=False)
    probs = torch.softmax(process_ref(logits[0], 0.8, 10, 0.9).double(), 0)
    freq = torch.bincount(tok, minlength=V).double() / n
    assert (freq - probs).abs().max() < 0.03
    assert freq[probs == 0].sum() == 0


@pytest.mark.gpu
def test_deterministic_and_graph_replay():
    from gpu_utils import graph_replays_match
    from acorninfer_amd.sampler import sample_batch
    logits = _rows(4, 151936, torch.bfloat16, 13).cuda()
    t = torch.tensor([0.7, 1.0, 0.0, 1.2], device="cuda")
    k = torch.tensor([20, 0, 0, 100], dtype=torch.int32, device="cuda")
    p = torch.tensor([0.95, 0.9, 1.0, 0.8], device="cuda")
    u = torch.tensor([0.1, 0.5, 0.9, 0.33], device="cuda")
    tok = torch.empty(4, dtype=torch.int64, device="cuda")
    lp = torch.empty(4, device="cuda")
    st = torch.empty(4, dtype=torch.int32, device="cuda")

    def run():
        sample_batch(logits, t, k, p, u, token=tok, logprob=lp, status=st)
    run()
    first = tok.clone()
    run()
    assert torch.equal(first, tok)
    assert graph_replays_match(run, lambda: tok)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [151936, 151935, 1000])
def test_greedy_is_first_maximum(dtype, V):
    """Temperature 0 against torch.argmax (first maximal index) on rows built
    to tie: the maximum in several 16-byte vectors of one thread and of
    different threads, twice inside one vector, +0/-0 as the maximum, in the
    scalar tail, and a constant row. An odd V puts every other row off
    16-byte alignment (the kernel's scalar path) and leaves a tail."""
    from acorninfer_amd.sampler import sample_batch
    E = 16 // torch.tensor([], dtype=dtype).element_size()   # elements per 16-byte vector
    g = torch.Generator().manual_seed(V)
    x = (torch.randn(6, V, generator=g) * 3).clamp(-20, 20)
    top = 40.0
    for i in [9001, 5 * E + 3, (5 + 1024) * E, 7 * E + E - 1]:   # same thread / other threads
        if i < V:
            x[1, i] = top
    x[2, 3 * E + 1] = top                                        # twice in one vector
    x[2, 3 * E + E - 1] = top
    x[3] = -x[3].abs() - 1.0                                     # the maximum is a zero
    x[3, 50] = 0.0
    x[3, 100] = -0.0
    x[3, 20] = -0.0
    x[4, V - 1] = top                                            # last element, and earlier
    x[4, V // 3] = top
    x[5] = 1.0                                                   # constant row
    logits = x.to(dtype)
    B = logits.shape[0]
    zeros = torch.zeros(B, device="cuda")
    tok, lp, st = sample_batch(logits.cuda(), zeros, torch.zeros(B, dtype=torch.int32,
                                                                   device="cuda"),
                               torch.ones(B, device="cuda"), zeros)
    assert st.cpu().eq(0).all()
    want = torch.argmax(logits.float(), dim=1)
    assert tok.cpu().tolist() == want.tolist()
    assert lp.cpu().eq(0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [16384, 16385, 16640 + 9, 151936])
def test_split_rows_equal_one_workgroup_rows(dtype, V):
    """The split form (a workspace given) against the one-workgroup form
    (acorn_sample) on the same rows: the kept set and its values bit for bit,
    the token the one whose interval of the 64-bit cumulative distribution holds
    the uniform, the logprob within fp32 rounding. V: the shortest split
    row, odd lengths (rows off 16-byte alignment, a short last chunk), a
    vocabulary. Rows: peaked, flat, all equal (every element on the boundary:
    handed to the one-workgroup form), few distinct values (ties across
    chunks), a tie group of the maximum, zeros of both signs, a maximum in the
    last element, an infinity. Options: each of top-k and top-p alone,
    together, neither, a top-k past the lists (of the row, of a chunk), greedy, a
    tiny top-p."""
    from acorninfer_amd._lib import check, dtype_code, lib, ptr, stream_ptr
    from acorninfer_amd.sampler import sample_batch, sample_workspace
    g = torch.Generator().manual_seed(V)
    x = torch.randn(8, V, generator=g) * 3
    x[0, ::997] += 9
    x[2] = 1.5
    x[3] = torch.randint(0, 40, (V,), generator=g).float() / 8
    x[4, ::V // 40] = 15.0
    x[5] = -x[5].abs()
    x[5, ::777] = 0.0
    x[5, 5::777] = -0.0
    x[6, V - 1] = 30.0
    x[7, V // 2] = float("inf")
    options = [(0.7, 20, 0.95), (1.0, 0, 0.9), (0.6, 50, 1.0), (1.0, 0, 1.0), (0.9, 5000, 0.8),
               (0.0, 0, 1.0), (1.0, 1, 1.0), (1.2, 0, 1e-6), (0.8, V, 0.5), (1.1, 100, 0.9)]
    rows = x.repeat_interleave(len(options), 0).to(dtype).cuda()
    opts = options * x.shape[0]
    B = rows.shape[0]
    t = torch.tensor([o[0] for o in opts], device="cuda")
    k = torch.tensor([o[1] for o in opts], dtype=torch.int32, device="cuda")
    p = torch.tensor([o[2] for o in opts], device="cuda")
    u = torch.rand(B, generator=g).cuda()
    assert sample_workspace(B, V, "cuda") is not None
    got_p, want_p = (torch.full((B, V), 7.0, device="cuda") for _ in range(2))
    tok, lp, st = sample_batch(rows, t, k, p, u, processed=got_p)
    wtok, wlp, wst = torch.empty_like(tok), torch.empty_like(lp), torch.empty_like(st)
    check(lib().acorn_sample(ptr(rows), B, V, dtype_code(rows), ptr(t), ptr(k), ptr(p), ptr(u),
                             ptr(wtok), ptr(wlp), ptr(want_p), ptr(wst), stream_ptr()), "sample")
    assert torch.equal(st, wst) and int(st.sum()) == len(options)
    assert torch.equal(got_p, want_p)
    drawn = (wst == 0) & (t > 0)
    assert torch.equal(tok[~drawn], wtok[~drawn])
    # the masses are exp2f of x - max (at most 28 in magnitude where they count)
    # times log2 e in fp32: within 28 * 2^-24 + 2 ulp, i.e. 2e-6, of exact
    prob = torch.softmax(want_p[drawn].double(), 1)
    cum = prob.cumsum(1).gather(1, tok[drawn, None])[:, 0]
    lo = cum - prob.gather(1, tok[drawn, None])[:, 0]
    assert (prob.gather(1, tok[drawn, None]) > 0).all()
    assert ((lo - 4e-6 <= u[drawn]) & (u[drawn] <= cum + 4e-6)).all()
    # sums of at most 151936 fp32 terms against exact integer sums
    same = tok == wtok
    assert same.float().mean() > 0.9
    torch.testing.assert_close(lp[same], wlp[same], rtol=1e-5, atol=1e-5, equal_nan=True)
    # without the processed row (no fifth launch), and twice
    for _ in range(2):
        tok2, lp2, _ = sample_batch(rows, t, k, p, u)
        assert torch.equal(tok2, tok) and torch.equal(lp2.view(torch.int32), lp.view(torch.int32))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [16384, 16640 + 9, 151936])
def test_split_rows_with_long_boundaries_equal_one_workgroup_rows(dtype, V):
    """Rows whose boundary holds more elements than the split form's lists (64 per
    chunk, 1024 per row), against the one-workgroup form as above: the kept set and
    its values bit for bit, the draw by the 64-bit distribution. Rows: logits of
    high magnitude (in bf16 one value is a tie group of more than 1024), flat ones,
    a spread within one bin, around 0 with both signs, two values, all equal but
    one, and ties only in the first and the last chunk. Options: top-p alone, high
    and low, a large top-k alone and with top-p, both at a T that widens or narrows
    the bins."""
    from acorninfer_amd._lib import check, dtype_code, lib, ptr, stream_ptr
    from acorninfer_amd.sampler import sample_batch
    g = torch.Generator().manual_seed(V + 1)
    x = torch.randn(8, V, generator=g)
    x[0] = x[0] * 2 + 8
    x[1] *= 0.1
    x[2] = 3 + x[2] * 1e-3
    x[3] *= 1e-5
    x[4] = torch.randint(0, 2, (V,), generator=g).float()
    x[5] = -4.0
    x[5, V // 3] = -1.0
    x[6] = -5 + 0.01 * x[6]
    x[6, :70] = 6.0
    x[6, V - 75:] = 6.0
    options = [(1.0, 0, 0.9), (0.3, 0, 0.5), (1.7, 0, 0.999), (1.0, 5000, 1.0), (0.8, 5000, 0.8),
               (1.3, V - 1, 0.3), (1.0, 100, 0.95), (1.0, 120, 0.4), (1.0, 0, 1e-6)]
    rows = x.repeat_interleave(len(options), 0).to(dtype).cuda()
    opts = options * x.shape[0]
    B = rows.shape[0]
    t = torch.tensor([o[0] for o in opts], device="cuda")
    k = torch.tensor([o[1] for o in opts], dtype=torch.int32, device="cuda")
    p = torch.tensor([o[2] for o in opts], device="cuda")
    u = torch.rand(B, generator=g).cuda()
    got_p, want_p = (torch.full((B, V), 7.0, device="cuda") for _ in range(2))
    tok, lp, st = sample_batch(rows, t, k, p, u, processed=got_p)
    wtok, wlp, wst = torch.empty_like(tok), torch.empty_like(lp), torch.empty_like(st)
    check(lib().acorn_sample(ptr(rows), B, V, dtype_code(rows), ptr(t), ptr(k), ptr(p), ptr(u),
                             ptr(wtok), ptr(wlp), ptr(want_p), ptr(wst), stream_ptr()), "sample")
    assert int(st.sum()) == 0 and int(wst.sum()) == 0
    assert torch.equal(got_p, want_p)
    # the drawn token's interval of the distribution holds the uniform (bounds as above)
    prob = torch.softmax(want_p.double(), 1)
    cum = prob.cumsum(1).gather(1, tok[:, None])[:, 0]
    lo = cum - prob.gather(1, tok[:, None])[:, 0]
    assert (prob.gather(1, tok[:, None]) > 0).all()
    assert ((lo - 4e-6 <= u) & (u <= cum + 4e-6)).all()
    same = tok == wtok
    torch.testing.assert_close(lp[same], wlp[same], rtol=1e-5, atol=1e-5)
    tok2, lp2, _ = sample_batch(rows, t, k, p, u)
    assert torch.equal(tok2, tok) and torch.equal(lp2, lp)


@pytest.mark.gpu
@pytest.mark.parametrize("V", [16384, 20003])
@pytest.mark.parametrize("B", [9, 16, 17, 40, 130, 600])
def test_split_forms_of_few_and_of_many_rows_agree(B, V):
    """Batches past 8 rows run their chunks on smaller workgroups and, past 16, the
    maxima of 2 to 32 chunks on one: every row's token, logprob and processed row are
    those it has in a batch of 8, bit for bit. Every option, a greedy and a
    non-finite row among them."""
    from acorninfer_amd.sampler import sample_batch
    g = torch.Generator().manual_seed(B)
    x = torch.randn(B, V, generator=g) * 3
    x[::5] *= 0.1
    x[3, V // 2] = float("inf")
    x[6, V - 1] = 40.0
    rows = x.bfloat16().cuda()
    options = [(0.7, 20, 0.95), (1.0, 0, 0.9), (0.6, 50, 1.0), (1.0, 0, 1.0), (0.9, 5000, 0.8),
               (0.0, 0, 1.0), (1.0, 1, 1.0)]
    opts = [options[i % len(options)] for i in range(B)]
    t = torch.tensor([o[0] for o in opts], device="cuda")
    k = torch.tensor([o[1] for o in opts], dtype=torch.int32, device="cuda")
    p = torch.tensor([o[2] for o in opts], device="cuda")
    u = torch.rand(B, generator=g).cuda()

    def run(s):
        proc = torch.full((s.stop - s.start, V), 7.0, device="cuda")
        return (*sample_batch(rows[s], t[s], k[s], p[s], u[s], processed=proc), proc)
    whole = run(slice(0, B))
    for a in range(0, B, 8):
        s = slice(a, min(a + 8, B))
        for got, want in zip(whole, run(s)):
            assert torch.equal(got[s].nan_to_num(99.0), want.nan_to_num(99.0)), s


def test_split_rows_are_those_whose_masses_add_up_in_64_bits():
    """The split form's sums (no GPU): a row of V equal logits has mass V x 2^40,
    which passes 2^64 from 2^24 elements; longer rows have no workspace and run
    on the one-workgroup form, whose draw adds in fp32."""
    import ctypes
    from acorninfer_amd._lib import check, lib
    n = ctypes.c_int64(-1)
    for V, split in ((16383, False), (16384, True), (151936, True), (1 << 23, True),
                     ((1 << 24) + 8, False), (1 << 31, False)):
        check(lib().acorn_sample_workspace(3, V, ctypes.byref(n)), "workspace")
        assert (n.value > 0) == split, V
        assert not split or V * 2 ** 40 < 2 ** 64
