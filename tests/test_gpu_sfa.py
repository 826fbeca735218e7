"""GPU parity of the sparse-attention consumer (kvip_hip_sparse_attention through
kvip_amd.sparse_attention) against oracle/sfa.py, on the reference's KV payload rows.

Bars: the reference's own tolerance for this check (allclose atol 0.006, rtol 0.025,
correctness.py:329-330) and, tighter, a maximum absolute error below 3e-3; rows with no
valid index give zeros; bad positions are reported in status. Three sources of rows: a paged
cache with random indices (8, 16, 24, 40, 72 and 128 heads: one head group per workgroup, two
groups sharing each staged tile (24: the second group partly filled), a set whose second group
holds no heads; absent and repeated
indices; and, with enough rows that no index split is needed, 256 rows at 16 heads and 128
rows at 128 heads, whose workgroups write the normalised output themselves), the gathered
buffer of the contiguous LIFetch forward, and the resident hot cache addressed by the slot
outputs (the reference's check_sfa flow: slots from the round, values from the logical
tokens' payload)."""
import ctypes

import numpy as np
import pytest

import kvip_amd
from kvip_amd import synthetic
from kvip_amd.operators.sfa import gathered_table, hot_cache_table, sparse_attention
from kvip_amd.runtime import abi
from oracle import sfa

pytestmark = pytest.mark.gpu
TOPK = 2048
ROW = 656
SCALE = 576 ** -0.5


def say(*args):
    print(*args, flush=True)


def bf16_query(torch, rng, rows, heads):
    q = rng.uniform(-0.2, 0.2, (rows, heads, 576)).astype(np.float32)
    qt = torch.from_numpy(q).to(torch.bfloat16)
    return qt.cuda(), qt.float().numpy()


def check(got, want, label):
    err = float(np.max(np.abs(got - want)))
    say(f"  {label}: max abs error {err:.2e}")
    assert np.all(np.isfinite(got)), label
    assert np.allclose(got, want, atol=0.006, rtol=0.025), (label, err)
    assert err < 3e-3, (label, err)


@pytest.mark.parametrize("heads,rpr", [(8, 1), (16, 2), (24, 1), (40, 4), (72, 2), (128, 1)])
def test_sparse_attention_paged_matches_oracle(torch_gpu, heads, rpr):
    torch = torch_gpu
    rng = np.random.default_rng(heads)
    say(f"case paged heads={heads} rows_per_request={rpr}")
    blocks, max_blocks, rows = 48, 24, 8
    batch = rows // rpr
    h_kv = np.concatenate([sfa.kv_payload(int(b % 5), np.arange(128) + b * 128) for b in range(blocks)])
    h_kv = h_kv.reshape(blocks, 128, ROW)
    table = np.stack([rng.permutation(blocks)[:max_blocks] for _ in range(batch)]).astype(np.int32)
    idx = rng.integers(0, max_blocks * 128, (rows, TOPK)).astype(np.int32)
    idx[rng.random((rows, TOPK)) < 0.2] = -1
    idx[1, 100:300] = idx[1, 0]  # a repeated position counts every time
    idx[rows - 1] = -1           # no valid index: zeros
    q, qh = bf16_query(torch, rng, rows, heads)
    out = sparse_attention(q, torch.from_numpy(h_kv).cuda(), torch.from_numpy(table).cuda(),
                           torch.from_numpy(idx).cuda(), SCALE, rows_per_request=rpr).cpu().numpy()
    want = np.zeros((rows, heads, 512), np.float32)
    for r in range(rows - 1):
        t = idx[r][idx[r] >= 0]
        want[r] = sfa.sparse_attention(qh[r], h_kv[table[r // rpr][t // 128], t % 128], SCALE)
    check(out, want, f"paged h{heads}")
    assert not out[rows - 1].any()


@pytest.mark.parametrize("heads,rows", [(16, 256), (128, 128)])
def test_sparse_attention_unsplit_rows_match_oracle(torch_gpu, heads, rows):
    """Enough rows that the launch fills the GPU without index splits: each workgroup
    normalises and writes its heads' output itself (no partials, no merge launch), for
    the 16-head kernel and for the kernel of four waves per 32 heads."""
    torch = torch_gpu
    rng = np.random.default_rng(heads + rows)
    say(f"case unsplit heads={heads} rows={rows}")
    blocks, max_blocks = 40, 20
    h_kv = np.concatenate([sfa.kv_payload(int(b % 3), np.arange(128) + b * 128) for b in range(blocks)])
    h_kv = h_kv.reshape(blocks, 128, ROW)
    table = np.stack([rng.permutation(blocks)[:max_blocks] for _ in range(rows)]).astype(np.int32)
    idx = rng.integers(0, max_blocks * 128, (rows, TOPK)).astype(np.int32)
    idx[rng.random((rows, TOPK)) < 0.75] = -1
    q, qh = bf16_query(torch, rng, rows, heads)
    out = sparse_attention(q, torch.from_numpy(h_kv).cuda(), torch.from_numpy(table).cuda(),
                           torch.from_numpy(idx).cuda(), SCALE).cpu().numpy()
    for r in range(rows):
        t = idx[r][idx[r] >= 0]
        want = sfa.sparse_attention(qh[r], h_kv[table[r][t // 128], t % 128], SCALE)
        if r % 32 == 0:
            say(f"  row {r}: max abs error {float(np.max(np.abs(out[r] - want))):.2e}")
        assert np.all(np.isfinite(out[r])), r
        assert np.allclose(out[r], want, atol=0.006, rtol=0.025), r
        assert float(np.max(np.abs(out[r] - want))) < 3e-3, r


def test_sparse_attention_reports_bad_positions(torch_gpu):
    torch = torch_gpu
    rng = np.random.default_rng(2)
    h_kv = sfa.kv_payload(0, np.arange(4 * 128)).reshape(4, 128, ROW)
    table = np.array([[0, 1, 2, 3], [3, 2, 1, 9]], np.int32)  # block 9 does not exist
    idx = rng.integers(0, 512, (2, TOPK)).astype(np.int32)
    idx[0, 5] = 512    # beyond the block table
    idx[1, :] = 400    # block 3 of request 1 -> 9: absent throughout
    q, qh = bf16_query(torch, rng, 2, 8)
    op = kvip_amd.SparseAttention(torch, rows=2, heads=8, device="cuda")
    op.bind(q, torch.from_numpy(h_kv).cuda(), torch.from_numpy(table).cuda(), torch.from_numpy(idx).cuda(), SCALE)
    out = op().cpu().numpy()
    torch.cuda.synchronize()
    status = int(op.status.item())
    assert status & abi_bits("BAD_TOKEN") and status & abi_bits("BAD_BLOCK"), status
    keep = np.delete(idx[0], 5)
    check(out[:1], sfa.sparse_attention(qh[0], h_kv[table[0][keep // 128], keep % 128], SCALE)[None], "bad-row")
    assert not out[1].any()


def abi_bits(name):
    from kvip_amd.runtime import abi
    return getattr(abi, f"STATUS_{name}")


def test_sparse_attention_on_gathered_rows(torch_gpu):
    torch = torch_gpu
    say("case gathered rows of the contiguous forward")
    wl = synthetic.decode_workload(torch, batch=4, ctx=[9000, 2100, 5000, 3000], device="cuda", seed=3)
    blocks = int(wl.kv_cache.shape[0])
    h_kv = np.concatenate([sfa.kv_payload(int(b % 7), np.arange(128) + b * 128) for b in range(blocks)])
    wl.kv_cache.copy_(torch.from_numpy(h_kv.reshape(blocks, 128, ROW)))
    rot, upd, fwd = synthetic.bind(torch, kvip_amd, wl)
    fwd()
    torch.cuda.synchronize()
    kv, table, indices = gathered_table(torch, upd)
    rng = np.random.default_rng(9)
    q, qh = bf16_query(torch, rng, 4, 16)
    out = sparse_attention(q, kv, table, indices, SCALE).cpu().numpy()
    top = rot.topk.cpu().numpy()
    bt = wl.block_table.cpu().numpy()
    h_kv = h_kv.reshape(blocks, 128, ROW)
    want = np.stack([sfa.sparse_attention(qh[r], h_kv[bt[r][top[r] // 128], top[r] % 128], SCALE) for r in range(4)])
    check(out, want, "gathered")


def test_sparse_attention_on_resident_hot_cache(torch_gpu):
    """check_sfa (correctness.py:261-339): LI + TopK + resident round on the device, then
    attention over the hot cache at the slot outputs against the logical tokens' payload."""
    torch = torch_gpu
    say("case resident hot cache")
    batch, owners, history, resident, q_rows = 2, 2, 8192, 4096, 4
    rng = np.random.default_rng(21)
    keys = rng.integers(0, 256, (owners, history, 128), dtype=np.uint8) & 0x77
    pool = np.concatenate([sfa.kv_payload(o, np.arange(history)) for o in range(owners)])
    t, dev = torch, "cuda"
    pool_t = t.empty(pool.size, dtype=t.uint8, pin_memory=True)
    pool_t.copy_(t.from_numpy(pool.reshape(-1)))
    hot = t.from_numpy(np.stack([pool[o * history:o * history + resident] for o in range(owners)])).to(dev)
    rot = kvip_amd.LIFetchBinding(t, batch=batch, max_context=history, device=dev, heads=32, rows_per_request=q_rows,
                                  qk_dtype="fp8", query_ends=True)
    rot.seq_lens.fill_(history)
    rot.query_ends.copy_(t.arange(history - 3, history + 1, dtype=t.int32).repeat(batch))
    # The four MTP rows of a request share their LI query, so their selections overlap and
    # the misses fit the LRU candidates.
    q_li = np.repeat(rng.standard_normal((batch, 32, 128)).astype(np.float32), q_rows, axis=0)
    rot.query.copy_(t.from_numpy(q_li).to(t.float8_e4m3fn))
    rot.weights.copy_(t.from_numpy(np.repeat(rng.standard_normal((batch, 32)).astype(np.float32), q_rows, axis=0)))
    upd = kvip_amd.ResidentIndexUpdate(
        t, keys=t.from_numpy(keys).to(dev).view(t.float8_e4m3fn),
        scales=t.from_numpy(rng.uniform(0.5, 2.0, (owners, history)).astype(np.float32)).to(dev),
        addresses=t.from_numpy((np.arange(owners * history) * ROW).reshape(owners, history)).to(dev),
        logical_ids=t.arange(history, dtype=t.int64, device=dev).repeat(owners, 1).contiguous(),
        row_owners=t.arange(batch, dtype=t.int32, device=dev), rotating=rot,
        hot_valid=t.ones((owners, resident), dtype=t.int32, device=dev), hot_cache=hot, host_pool=pool_t,
        resident=resident)
    upd.set_candidates(t.from_numpy(np.stack([rng.permutation(resident)[:TOPK] for _ in range(batch)])
                                    .astype(np.int32)).to(dev))
    kvip_amd.LIFetch(rot, upd)()
    t.cuda.synchronize()
    assert not upd.status.any(), upd.status.cpu().tolist()
    kv, table = hot_cache_table(t, upd)
    q, qh = bf16_query(t, rng, batch * q_rows, 8)
    out = sparse_attention(q, kv, table, upd.slot_output.view(batch * q_rows, TOPK), SCALE,
                           rows_per_request=q_rows).cpu().numpy()
    logical = upd.logical_output.view(batch * q_rows, TOPK).cpu().numpy()
    assert (logical >= 0).all()
    want = np.stack([sfa.sparse_attention(qh[r], sfa.kv_payload(r // q_rows, logical[r]), SCALE)
                     for r in range(batch * q_rows)])
    check(out, want, "resident hot cache")


@pytest.mark.parametrize("heads", [16, 128])
def test_sparse_attention_graph_replay(torch_gpu, heads):
    """The split launch and its merge launch captured in a hipGraph (the 16-head kernel and
    the kernel of four waves per 32 heads): every replay, with eager work between replays,
    equals the eager call bit for bit, and so does an eager call after the replays."""
    torch = torch_gpu
    rng = np.random.default_rng(33)
    rows, blocks = 16, 40
    h_kv = np.concatenate([sfa.kv_payload(int(b % 3), np.arange(128) + b * 128) for b in range(blocks)])
    kv = torch.from_numpy(h_kv.reshape(blocks, 128, ROW)).cuda()
    table = torch.from_numpy(np.stack([rng.permutation(blocks)[:16] for _ in range(rows)]).astype(np.int32)).cuda()
    idx = torch.from_numpy(rng.integers(0, 16 * 128, (rows, TOPK)).astype(np.int32)).cuda()
    q, _ = bf16_query(torch, rng, rows, heads)
    op = kvip_amd.SparseAttention(torch, rows=rows, heads=heads, device="cuda").bind(q, kv, table, idx, SCALE)
    eager = op().clone()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph):
            op()
    torch.cuda.current_stream().wait_stream(side)
    for replay in range(3):
        op.output.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(op.output, eager), replay
        _ = (q.float() * 2).sum().item()  # eager work between replays
    op.output.zero_()
    assert torch.equal(op(), eager)


@pytest.mark.parametrize("heads,rows,per_request", [(1, 1, 1), (16, 3, 1), (17, 40, 2), (33, 6, 1), (48, 200, 4)])
def test_sparse_attention_edges_against_64_bits(torch_gpu, heads, rows, per_request):
    """Partly filled head groups and sets, every split count (16 splits for one row down to
    none for 200), rows with a single index, with whole tiles of absent indices and with
    all 2048, queries whose features span 2^-20 .. 2^3 within a scale group, and a cache whose
    block 0, row 0 (never selected) is NaN throughout. Each probability is rounded once to
    bf16 (2^-9 relative), everything else is fp32: the error is held to twice that bound,
    2^-8 sum_j p_j |v_j| / sum_j p_j per feature."""
    torch = torch_gpu
    gen = torch.Generator(device="cuda").manual_seed(heads * 1000 + rows)
    batch, max_blocks = rows // per_request, 20
    blocks = 64
    values = torch.randn((blocks * 128, 4, 128), generator=gen, device="cuda")
    scales = torch.rand((blocks * 128, 4), generator=gen, device="cuda") * 0.02 + 0.0005
    kv = torch.empty((blocks * 128, ROW), dtype=torch.uint8, device="cuda")
    codes = (values * 60).to(torch.float8_e4m3fn)
    kv[:, :512] = codes.view(torch.uint8).view(-1, 512)
    rope = torch.randn((blocks * 128, 64), generator=gen, device="cuda").to(torch.bfloat16)
    kv[:, 512:640] = rope.view(torch.uint8)
    kv[:, 640:] = scales.view(torch.uint8)
    kv[0] = 0x7F  # NaN codes; rope and scales 0x7F7F..: huge
    kv[0, 640:] = torch.full((4,), float("nan"), device="cuda").view(torch.uint8)
    table = torch.stack([torch.randperm(blocks - 1, generator=gen, device="cuda")[:max_blocks] + 1 for _ in range(batch)])
    table = table.to(torch.int32)
    idx = torch.randint(0, max_blocks * 128, (rows, TOPK), generator=gen, device="cuda", dtype=torch.int32)
    idx[0, 1:] = -1
    if rows > 1:
        idx[1, 64:1024] = -1
        idx[1, 1500::3] = -1
    span = torch.randint(-20, 4, (rows, heads, 576), generator=gen, device="cuda").float()
    q = (torch.randn((rows, heads, 576), generator=gen, device="cuda") * torch.exp2(span)).to(torch.bfloat16)
    say(f"case edges heads={heads} rows={rows}")
    out = sparse_attention(q, kv.view(blocks, 128, ROW), table, idx, SCALE, rows_per_request=per_request).double()
    key = torch.cat([(codes.double() * scales.double()[:, :, None]).view(-1, 512), rope.double()], dim=1)
    worst = 0.0
    for r in sorted({0, 1 % rows, rows // 2, rows - 1}):
        t = idx[r][idx[r] >= 0].long()
        k = key[table[r // per_request].long()[t // 128] * 128 + t % 128].contiguous()
        prob = torch.softmax(q[r].double() @ k.T.contiguous() * SCALE, dim=1)
        want = prob @ k[:, :512].contiguous()
        bound = 2.0 ** -8 * (prob @ k[:, :512].abs().contiguous()) + 1e-7
        worst = max(worst, ((out[r] - want).abs() / bound).max().item())
    say(f"  worst error over its bound: {worst:.3f}")
    assert worst <= 1.0


@pytest.mark.parametrize("heads,rows,spread", [
    (16, 3, "span"), (40, 5, "span"), (128, 64, "span"), (16, 3, 10), (16, 64, 14), (40, 5, 12), (40, 5, 20),
    (128, 64, 16), (8, 200, 60)])
def test_sparse_attention_query_spread_against_64_bits(torch_gpu, heads, rows, spread):
    """Queries whose large features meet zero key bytes, so that the logits are made of the small ones.
    "span": features down to 2^-13 of their scale group's largest, the bytes zero at those above
    2^-6. A number k: one feature of groups 0 and 2 of the first 16 heads is 2^k times the
    others and meets zero bytes. The logits are scaled to a standard deviation of 3, so an error in
    them shows in the output. The bound is that of the test above: one bf16 rounding per
    probability, doubled."""
    torch = torch_gpu
    gen = torch.Generator(device="cuda").manual_seed(heads * 100 + rows)
    blocks, max_blocks = 64, 20
    q = torch.randn((rows, heads, 576), generator=gen, device="cuda")
    codes = (torch.randn((blocks * 128, 4, 128), generator=gen, device="cuda") * 60).to(torch.float8_e4m3fn)
    if spread == "span":
        at = torch.arange(512, device="cuda") % 14  # power of two below the largest
        q[:, :, :512] = (1 + torch.rand((rows, heads, 512), generator=gen, device="cuda")) * torch.exp2(6.0 - at)
        q[:, :, :512] *= torch.where(torch.rand((rows, heads, 512), generator=gen, device="cuda") < 0.5, -1.0, 1.0)
        q = torch.where(q.to(torch.bfloat16).abs() >= 128, 127.5, q)  # no value rounds into the next power of two
        codes.view(torch.uint8).view(-1, 512)[:, at < 6] = 0
    else:
        for feature in (17, 300):
            q[:, :16, feature] = 1.37 * 2.0 ** spread
            codes.view(torch.uint8).view(-1, 512)[:, feature] = 0
    q = q.to(torch.bfloat16)
    scales = torch.rand((blocks * 128, 4), generator=gen, device="cuda") * 0.01 + 0.01
    rope = torch.randn((blocks * 128, 64), generator=gen, device="cuda").to(torch.bfloat16)
    kv = torch.empty((blocks * 128, ROW), dtype=torch.uint8, device="cuda")
    kv[:, :512] = codes.view(torch.uint8).view(-1, 512)
    kv[:, 512:640] = rope.view(torch.uint8)
    kv[:, 640:] = scales.view(torch.uint8)
    table = torch.stack([torch.randperm(blocks, generator=gen, device="cuda")[:max_blocks] for _ in range(rows)])
    table = table.to(torch.int32)
    idx = torch.randint(0, max_blocks * 128, (rows, TOPK), generator=gen, device="cuda", dtype=torch.int32)
    key = torch.cat([(codes.double() * scales.double()[:, :, None]).view(-1, 512), rope.double()], dim=1)
    picked = {r: key[table[r].long()[idx[r].long() // 128] * 128 + idx[r].long() % 128].contiguous()
              for r in sorted({0, rows // 2, rows - 1})}
    scale = 3.0 / (q[0].double() @ picked[0].T.contiguous()).std().item()
    say(f"case query spread heads={heads} rows={rows} spread={spread} scale={scale:.4f}")
    out = sparse_attention(q, kv.view(blocks, 128, ROW), table, idx, scale).double()
    worst = 0.0
    for r, k in picked.items():
        prob = torch.softmax(q[r].double() @ k.T.contiguous() * scale, dim=1)
        bound = 2.0 ** -8 * (prob @ k[:, :512].abs().contiguous()) + 1e-7
        worst = max(worst, ((out[r] - prob @ k[:, :512].contiguous()).abs() / bound).max().item())
    say(f"  worst error over its bound: {worst:.3f}")
    assert worst <= 1.0


@pytest.mark.parametrize("heads", [16, 40])
def test_sparse_attention_nonfinite_query_stays_in_its_head(torch_gpu, heads):
    """A NaN feature makes its head NaN. An infinite one that meets only negative key bytes makes every
    logit of its head -inf, and that head is zero. The other heads are as without them."""
    torch = torch_gpu
    gen = torch.Generator(device="cuda").manual_seed(heads)
    rows, blocks = 2, 32
    kv = torch.zeros((blocks * 128, ROW), dtype=torch.uint8, device="cuda")
    codes = (torch.randn((blocks * 128, 512), generator=gen, device="cuda") * 60).to(torch.float8_e4m3fn)
    codes.view(torch.uint8)[:, 200] = 0xB8  # -1
    kv[:, :512] = codes.view(torch.uint8)
    kv[:, 640:] = torch.full((4,), 0.02, device="cuda").view(torch.uint8)
    table = torch.arange(blocks, dtype=torch.int32, device="cuda").expand(rows, blocks).contiguous()
    idx = torch.randint(0, blocks * 128, (rows, TOPK), generator=gen, device="cuda", dtype=torch.int32)
    q = torch.randn((rows, heads, 576), generator=gen, device="cuda").to(torch.bfloat16)
    say(f"case nonfinite query heads={heads}")
    want = sparse_attention(q, kv.view(blocks, 128, ROW), table, idx, SCALE).clone()
    q[:, 3, 5], q[:, 4, 200] = float("nan"), float("inf")
    out = sparse_attention(q, kv.view(blocks, 128, ROW), table, idx, SCALE)
    say("  infinite head:", out[:, 4].unique()[:4].tolist())
    assert out[:, 3].isnan().all() and (out[:, 4] == 0).all()
    others = [h for h in range(heads) if h not in (3, 4)]
    err = (out[:, others] - want[:, others]).abs().max().item()
    say(f"  other heads: max abs difference {err:.2e}")
    assert err <= 2.0 ** -8 * 448 * 0.02 / 4  # p rounded once to bf16, |v| mostly far below its largest


@pytest.mark.parametrize("rows,heads", [(2, 16), (3, 40), (260, 16)])
def test_sparse_attention_buffers_of_any_float_alignment(torch_gpu, rows, heads):
    """Output and workspace (16 splits for few rows, none for 260) 4 bytes past a 16-byte boundary: the
    same output, bit for bit, and nothing written beside it."""
    torch = torch_gpu
    gen = torch.Generator(device="cuda").manual_seed(rows)
    blocks = 24
    kv = torch.zeros((blocks, 128, ROW), dtype=torch.uint8, device="cuda")
    kv[:, :, :512] = torch.randint(0, 120, (blocks, 128, 512), generator=gen, device="cuda", dtype=torch.uint8)
    kv[:, :, 640:] = torch.full((4,), 0.01, device="cuda").view(torch.uint8)
    table = torch.arange(blocks, dtype=torch.int32, device="cuda").expand(rows, blocks).contiguous()
    idx = torch.randint(0, blocks * 128, (rows, TOPK), generator=gen, device="cuda", dtype=torch.int32)
    q = torch.randn((rows, heads, 576), generator=gen, device="cuda").to(torch.bfloat16)
    op = kvip_amd.SparseAttention(torch, rows=rows, heads=heads, device="cuda").bind(q, kv, table, idx)
    say(f"case float alignment rows={rows} heads={heads}")
    want = op().clone()
    out = torch.full((want.numel() + 8,), 7.0, device="cuda")
    work = torch.empty(op.workspace.numel() + 4, device="cuda")
    args = abi.SparseAttnArgs.from_buffer_copy(op.args)
    args.output, args.workspace = out[1:].data_ptr(), work[1:].data_ptr()
    assert args.output % 16 == 4 and args.workspace % 16 == 4
    assert op.library.kvip_hip_sparse_attention(ctypes.byref(args), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(out[1:1 + want.numel()].view_as(want), want)
    assert out[0] == 7 and (out[1 + want.numel():] == 7).all()
