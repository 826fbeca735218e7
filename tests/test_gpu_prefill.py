"""GPU parity of the prefill lightning indexer (kvip_hip_indexer_prefill + TopK) against
the CPU oracle, through the C ABI.

Bars: scores within 3e-2 relative for fp8 and 1e-2 for bf16 Q/K (each with an absolute
floor of that fraction of the row's largest |score|) and at least 99 % of the keys with |score| >= 3e-2 of the row's largest
bit-identical (fp8 MFMA dot products are not correctly rounded, so scores that cancel to
near zero differ in their last bits more often; measured 0.3 % there); visible lengths and the
high-byte histogram exact; TopK bit-exact against the oracle's TopK of the GPU's own
keys and inside the oracle's one-ulp cutoff band."""
import numpy as np
import pytest

import kvip_amd
from kvip_amd import synthetic
from oracle import indexer as ref

pytestmark = pytest.mark.gpu


def say(*args):
    print(*args, flush=True)


def make_case(torch, *, q_lens, k_lens, heads, wdt, qscale, kscale, seed, qk="fp8"):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rows = int(sum(q_lens))
    max_blocks = max((k + 127) // 128 for k in k_lens)
    blocks = sum((k + 127) // 128 for k in k_lens) + 3

    def operand(shape):
        x = torch.randn(shape, generator=g, device="cuda")
        return synthetic.saturating_fp8(torch, x) if qk == "fp8" else x.to(torch.bfloat16)

    keys = operand((blocks, 128, 128))
    key_scale = (torch.rand((blocks, 128), generator=g, device="cuda") * 1.5 + 0.5) if kscale else None
    query = operand((rows, heads, 128))
    weights = (torch.randn((rows, heads), generator=g, device="cuda") / 8).to(wdt)
    query_scale = (torch.rand((rows, heads), generator=g, device="cuda") + 0.5) if qscale else None
    perm = torch.randperm(blocks, generator=torch.Generator().manual_seed(seed)).int()
    table = torch.zeros((len(k_lens), max_blocks), dtype=torch.int32)
    at = 0
    for s, k in enumerate(k_lens):
        nb = (k + 127) // 128
        table[s, :nb] = perm[at:at + nb]
        at += nb
    cu = torch.tensor(np.concatenate([[0], np.cumsum(q_lens)]), dtype=torch.int32)
    kl = torch.tensor(k_lens, dtype=torch.int32)
    return dict(query=query, weights=weights, query_scale=query_scale, keys=keys, key_scale=key_scale,
                table=table.cuda(), cu=cu.cuda(), kl=kl.cuda(), rows=rows, max_ctx=max_blocks * 128)


def host(torch, t):
    if t is None:
        return None
    if t.dtype == torch.float8_e4m3fn:
        return ref.fp8_e4m3_decode(t.view(torch.uint8).cpu().numpy())
    return t.float().cpu().numpy()


CASES = [
    # name, q_lens, k_lens, heads, weight dtype, qscale, kscale, Q/K dtype
    ("h64_two_seqs", [37, 100], [3000, 5000], 64, "f32", True, True, "fp8"),
    ("h32_bf16w_short_ctx", [20, 5, 64], [300, 2, 4096], 32, "bf16", False, True, "fp8"),
    ("h64_more_rows_than_keys", [300], [260], 64, "f32", False, False, "fp8"),
    ("h64_long_rows", [64], [9000], 64, "f32", True, True, "fp8"),
    ("bf16qk_h64_two_seqs", [37, 100], [3000, 5000], 64, "f32", False, False, "bf16"),
    ("bf16qk_h32_scaled_short_ctx", [20, 5, 64], [300, 2, 4096], 32, "bf16", True, True, "bf16"),
    ("bf16qk_h64_long_rows", [64], [9000], 64, "f32", False, True, "bf16"),
    ("bf16qk_h64_more_rows_than_keys", [300], [260], 64, "bf16", True, False, "bf16"),
]


@pytest.mark.parametrize("name,q_lens,k_lens,heads,wdt,qscale,kscale,qk", CASES, ids=[c[0] for c in CASES])
def test_prefill_matches_oracle(torch_gpu, name, q_lens, k_lens, heads, wdt, qscale, kscale, qk):
    torch = torch_gpu
    say(f"case prefill {name}")
    c = make_case(torch, q_lens=q_lens, k_lens=k_lens, heads=heads,
                  wdt=torch.float32 if wdt == "f32" else torch.bfloat16, qscale=qscale, kscale=kscale, seed=17,
                  qk=qk)
    tol = 3e-2 if qk == "fp8" else 1e-2
    idx = kvip_amd.PrefillIndexer(torch, max_rows=c["rows"] + 5, max_context=c["max_ctx"],
                                  max_sequences=len(q_lens), device="cuda", heads=heads,
                                  weight_dtype=c["weights"].dtype)
    top = idx(c["query"], c["weights"], c["query_scale"], c["keys"], c["key_scale"], c["cu"], c["kl"], c["table"])
    torch.cuda.synchronize()
    assert int(idx.status.item()) == 0
    want, vis = ref.prefill_keys_paged(host(torch, c["query"]), host(torch, c["weights"]),
                                       host(torch, c["query_scale"]), host(torch, c["keys"]),
                                       host(torch, c["key_scale"]), c["table"].cpu().numpy(), c["cu"].cpu().numpy(),
                                       c["kl"].cpu().numpy(), idx.key_stride)
    assert np.array_equal(idx.row_valid[:c["rows"]].cpu().numpy(), vis)
    got = idx.score_keys[:c["rows"]].cpu().numpy().view(np.uint16)
    for r, v in enumerate(vis):
        if v == 0:
            continue
        gv = ref.score_values(got[r, :v]).astype(np.float64)
        wv = ref.score_values(want[r, :v]).astype(np.float64)
        bad = np.abs(gv - wv) > tol * np.abs(wv) + tol * np.abs(wv).max()
        assert not bad.any(), (r, int(bad.sum()))
    same = ref.identical_share(got, want, vis)
    say(f"  identical keys (|score| >= 3e-2 of row max): {same:.5f}")
    assert same > 0.99
    # TopK consumed and re-zeroed the histogram; it equals the oracle's TopK of the GPU keys.
    assert not idx.histogram.any()
    top = top.cpu().numpy()
    for r, v in enumerate(vis):
        assert np.array_equal(top[r], ref.topk_reference(got[r], v)), r
        if v >= 2048:
            assert ref.validate_topk_band(top[r], ref.score_values(want[r, :v])), r


def test_prefill_histogram_before_topk(torch_gpu):
    torch = torch_gpu
    c = make_case(torch, q_lens=[50, 30], k_lens=[4000, 700], heads=64, wdt=torch.float32, qscale=False,
                  kscale=True, seed=3)
    idx = kvip_amd.PrefillIndexer(torch, max_rows=c["rows"], max_context=c["max_ctx"], max_sequences=2,
                                  device="cuda")
    import ctypes
    from kvip_amd.runtime import abi
    p = abi.ptr
    args = abi.PrefillArgs(query=p(c["query"]), weights=p(c["weights"]), query_scale=0, keys=p(c["keys"]),
                           key_scale=p(c["key_scale"]), block_table=p(c["table"]), cu_seqlens_q=p(c["cu"]),
                           seq_lens_k=p(c["kl"]), score_keys=p(idx.score_keys), histogram=p(idx.histogram),
                           row_valid=p(idx.row_valid), status=p(idx.status), key_block_stride=c["keys"].stride(0),
                           scale_block_stride=c["key_scale"].stride(0), sequences=2, rows=c["rows"], heads=64,
                           max_blocks=int(c["table"].shape[1]), num_blocks=int(c["keys"].shape[0]),
                           key_stride=idx.key_stride, qk_dtype=abi.DTYPE_FP8_E4M3, weight_dtype=abi.DTYPE_FP32)
    abi.check(idx.library.kvip_hip_indexer_prefill(ctypes.byref(args), abi.stream_handle(torch, idx.device)), "LI")
    torch.cuda.synchronize()
    keys = idx.score_keys.cpu().numpy().view(np.uint16)
    hist = idx.histogram.cpu().numpy()
    for r, v in enumerate(idx.row_valid.cpu().numpy()):
        assert np.array_equal(hist[r], np.bincount(keys[r, :v] >> 8, minlength=256)), r


@pytest.mark.parametrize("qk,workgroups", [("fp8", 3), ("fp8", 64), ("bf16", 5)])
def test_prefill_bounded_grid_equals_full_grid(torch_gpu, qk, workgroups):
    """kvip_hip_indexer_prefill_grid: workgroups striding over the work units (fewer than the
    units, several units each, across sequences and segments) give the full grid's keys,
    visible lengths, histograms and TopK bit for bit."""
    torch = torch_gpu
    say(f"case prefill grid {qk} workgroups={workgroups}")
    c = make_case(torch, q_lens=[37, 100, 9], k_lens=[3000, 9000, 40], heads=64, wdt=torch.float32, qscale=True,
                  kscale=True, seed=23, qk=qk)
    idx = kvip_amd.PrefillIndexer(torch, max_rows=c["rows"], max_context=c["max_ctx"], max_sequences=3,
                                  device="cuda")
    idx.bind(c["query"], c["weights"], c["query_scale"], c["keys"], c["key_scale"], c["cu"], c["kl"], c["table"])
    results = []
    for wg in (0, workgroups):
        idx.score_keys.fill_(-1)
        idx.row_valid.fill_(-1)
        idx.score(workgroups=wg)
        torch.cuda.synchronize()
        vis = idx.row_valid.cpu().numpy()
        keys = idx.score_keys.cpu().numpy().view(np.uint16)
        hist = idx.histogram.cpu().numpy().copy()
        top = idx.select().cpu().numpy()
        torch.cuda.synchronize()
        assert int(idx.status.item()) == 0
        results.append((vis, [keys[r, :v].copy() for r, v in enumerate(vis)], hist, top))
    (v0, k0, h0, t0), (v1, k1, h1, t1) = results
    assert np.array_equal(v0, v1)
    assert all(np.array_equal(a, b) for a, b in zip(k0, k1))
    assert np.array_equal(h0, h1) and np.array_equal(t0, t1)
    assert h0.sum() == v0.sum()


@pytest.mark.parametrize("qk", ["fp8", "bf16"])
@pytest.mark.parametrize("rows,k_len", [(2050, 9001), (600, 9100), (130, 19999), (1024, 2049), (16, 4097)])
def test_prefill_rows_do_not_depend_on_the_segment(torch_gpu, qk, rows, k_len):
    """The launch picks 256 to 4096 keys per work item by rows and context: 1024, 512, 512, 512 and
    256 here for fp8, 4096, 2048, 1024, 1024 and 256 for bf16. A sequence's last 9 rows scored alone (256 keys per item, few items) see the same keys as the
    same rows of the whole sequence, so keys, histograms and TopK are the same, bit for bit."""
    torch = torch_gpu
    say(f"case prefill segment {qk} rows={rows} k_len={k_len}")
    c = make_case(torch, q_lens=[rows], k_lens=[k_len], heads=64, wdt=torch.float32, qscale=True, kscale=True,
                  seed=41, qk=qk)

    def score(first):
        n = rows - first
        idx = kvip_amd.PrefillIndexer(torch, max_rows=n, max_context=c["max_ctx"], max_sequences=1, device="cuda")
        idx.bind(c["query"][first:], c["weights"][first:], c["query_scale"][first:], c["keys"], c["key_scale"],
                 torch.tensor([0, n], dtype=torch.int32, device="cuda"), c["kl"], c["table"])
        idx.score()
        torch.cuda.synchronize()
        keys, vis, hist = idx.score_keys.clone(), idx.row_valid.clone(), idx.histogram.clone()
        top = idx.select().clone()
        assert int(idx.status.item()) == 0
        return keys, vis, hist, top

    whole, last = score(0), score(rows - 9)
    assert torch.equal(whole[1], torch.arange(k_len - rows + 1, k_len + 1, device="cuda", dtype=torch.int32))
    assert torch.equal(whole[2].sum(1, dtype=torch.int32), whole[1])
    for q in range(9):
        r, n = rows - 9 + q, k_len - 8 + q
        assert torch.equal(whole[0][r, :n], last[0][q, :n])
    for a, b in zip(whole[1:], last[1:]):
        assert torch.equal(a[rows - 9:], b)


def test_quant_lightning_indexer_wrapper(torch_gpu):
    """The native-call surface: TND rows, cumulative query lengths, [blocks,128,1,128] keys."""
    torch = torch_gpu
    c = make_case(torch, q_lens=[16, 40], k_lens=[2500, 3100], heads=64, wdt=torch.float32, qscale=True,
                  kscale=True, seed=5)
    out = kvip_amd.quant_lightning_indexer(
        c["query"], c["keys"].view(-1, 128, 1, 128), c["weights"], c["query_scale"], c["key_scale"].view(-1, 128, 1),
        c["cu"][1:], c["kl"], c["table"])
    torch.cuda.synchronize()
    idx = kvip_amd.PrefillIndexer(torch, max_rows=c["rows"], max_context=c["max_ctx"], max_sequences=2,
                                  device="cuda")
    direct = idx(c["query"], c["weights"], c["query_scale"], c["keys"], c["key_scale"], c["cu"], c["kl"], c["table"])
    assert out.shape == (c["rows"], 1, 2048)
    assert torch.equal(out.view(c["rows"], 2048), direct)


@pytest.mark.parametrize("qk", ["fp8", "bf16"])
@pytest.mark.parametrize("q_lens,k_lens", [
    ([40], [256]), ([3, 300], [257, 700]), ([2] * 69 + [9], [130] * 69 + [6001]), ([5] * 300, [600] * 150 + [4097] + [600] * 149),
    ([8], [0])])
def test_prefill_with_block_tables_wider_than_the_sequences(torch_gpu, qk, q_lens, k_lens):
    """Tables of 65536 positions against tables of the longest sequence: workgroups whose segment lies
    past every sequence leave early (the longest is the last of 70 and in the middle of 300
    sequences here), and keys, visible lengths, histograms and TopK are the same, bit for bit."""
    torch = torch_gpu
    say(f"case wide tables {qk} sequences={len(q_lens)} longest={max(k_lens)}")
    c = make_case(torch, q_lens=q_lens, k_lens=k_lens, heads=64, wdt=torch.float32, qscale=True, kscale=True, seed=23,
                  qk=qk)

    def run(table, workgroups=0):
        idx = kvip_amd.PrefillIndexer(torch, max_rows=c["rows"], max_context=max(table.shape[1], 1) * 128,
                                      max_sequences=len(q_lens), device="cuda")
        idx.bind(c["query"], c["weights"], c["query_scale"], c["keys"], c["key_scale"], c["cu"], c["kl"], table)
        idx.score(workgroups)
        torch.cuda.synchronize()
        keys, vis, hist = idx.score_keys.clone(), idx.row_valid.clone(), idx.histogram.clone()
        top = idx.select().clone()
        assert int(idx.status.item()) == 0
        return keys, vis, hist, top

    tight = c["table"] if c["table"].shape[1] else torch.zeros((len(q_lens), 1), dtype=torch.int32, device="cuda")
    wide = torch.zeros((len(q_lens), 512), dtype=torch.int32, device="cuda")
    wide[:, :tight.shape[1]] = tight
    want = run(tight)
    ends = np.concatenate([np.maximum(k - q + 1 + np.arange(q), 0) for q, k in zip(q_lens, k_lens)])
    assert np.array_equal(want[1].cpu().numpy(), ends)
    for got in (run(wide), run(wide, 100)):
        for a, b in zip(got[1:], want[1:]):
            assert torch.equal(a, b)
        for r, n in enumerate(ends):
            assert torch.equal(got[0][r, :n], want[0][r, :n])
