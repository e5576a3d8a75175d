"""Decode at f32 precision (f32 pages, head_dim other than 128, small scale
groups, GQA groups above 16) against the oracle's gather + flash_decode, at the
edges of its tiles: sequences around its 16-token tiles and the 64-tile windows
of a slice, head_dim below each built size, groups around its 16 heads, batches
around the 64 sequences of a scan step and on both sides of the 256 a wave scans
alone and of the 4096 of a launch, and the step's appended row."""
import numpy as np
import pytest

import airkv
from airkv import workloads
from gpu_helpers import log, rel_err, torch_mod
from test_gpu_decode import _decode_case
from test_gpu_decode_append import _run_pair, _setup

pytestmark = pytest.mark.gpu

# Both sides sum in f32 in orders of their own: at most n * 2^-24 apart for n
# <= 1100 keys (6.6e-5) relative to the largest output; half as much again
# covers the scores' own rounding.
TOL_F32 = 1e-4

LENS = [0, 14, 15, 16, 30, 31, 32, 62, 63, 64, 1, 255, 1022, 1024, 333]      # + 1 token each


# (dtype, head_dim, kv heads, group, block size, scale group, sequences)
CASES = [(dt, d, 2, 4, 16, 32, 15) for dt in (airkv.F32, airkv.BF16, airkv.INT8, airkv.FP8)
         for d in (32, 64, 96, 160, 256)] + [
    (airkv.F32, 128, 8, 1, 32, 32, 15), (airkv.F32, 128, 1, 17, 16, 32, 15), (airkv.BF16, 128, 1, 40, 32, 32, 15),
    (airkv.INT8, 128, 2, 7, 16, 16, 15), (airkv.FP8, 64, 2, 16, 32, 8, 15), (airkv.BF16, 224, 2, 16, 32, 32, 15),
    (airkv.F32, 192, 1, 3, 16, 32, 15), (airkv.FP8, 192, 2, 4, 32, 64, 15), (airkv.BF16, 64, 8, 4, 16, 32, 65), (airkv.F32, 64, 4, 2, 16, 32, 130), (airkv.INT8, 96, 1, 3, 32, 32, 64),
]


@pytest.mark.parametrize("q_bf16", [True, False])
@pytest.mark.parametrize("dtype,d,n_kv,group,bs,scale_group,batch", CASES)
def test_decode_f32_tile_edges(dtype, d, n_kv, group, bs, scale_group, batch, q_bf16):
    lens = (LENS * (batch // len(LENS) + 1))[:batch]
    cfg = workloads.Config("f32", n_kv * group, n_kv, d, bs, dtype, batch, scale_group=scale_group)
    got, want, (pool, host, tables, seq_lens, q, _) = _decode_case(cfg, lens, seed=13 + d + group, q_bf16=q_bf16)
    err = rel_err(got, want)
    # the same sequences in few, long slices, and in one
    torch = torch_mod()
    qt = torch.from_numpy(q).cuda()
    qt = qt.to(torch.bfloat16) if q_bf16 else qt
    for most in (1, 2, 7):
        out = torch.full(q.shape, float("nan"), device="cuda")
        pool.paged_decode(qt, torch.from_numpy(tables).cuda(), torch.from_numpy(seq_lens).cuda(), out, max_splits=most)
        err = max(err, rel_err(out.cpu().numpy(), want))
    log(f"decode f32 dtype={dtype} d={d} group={group} q_bf16={q_bf16}: rel err {err:.2e}")
    assert err <= TOL_F32
    assert pool.error_count() == 0


@pytest.mark.parametrize("dtype,d,n_q,scale_group", [(airkv.F32, 256, 20, 32), (airkv.BF16, 96, 7, 32),
                                                     (airkv.INT8, 160, 34, 32), (airkv.FP8, 32, 8, 8)])
def test_decode_f32_append_rows(dtype, d, n_q, scale_group):
    """The appended row at every place of a tile, 70 sequences: pages, scales
    and outputs equal append, then decode."""
    ctx = [i % 35 for i in range(70)]
    cfg = workloads.Config("f32", n_q, 1, d, 16, dtype, len(ctx), scale_group=scale_group)
    w, pa, pb, host, tables, lens, k_new, v_new = _setup(cfg, ctx, seed=7 + d)
    q = np.random.default_rng(8).standard_normal((len(ctx), n_q, d)).astype(np.float32)
    q, got = _run_pair(cfg, pa, pb, host, tables, lens, k_new, v_new, q, q_f32=True)
    assert rel_err(got, host.paged_decode(q, tables, lens, chunk=64)) <= TOL_F32


@pytest.mark.parametrize("dtype,d,n_kv,group,batch,bad", [
    (airkv.F32, 64, 1, 2, 255, 254), (airkv.BF16, 64, 2, 4, 256, 70), (airkv.INT8, 96, 1, 2, 257, 256),
    (airkv.BF16, 256, 2, 32, 400, 333), (airkv.F32, 32, 1, 1, 4100, 4098)])
def test_decode_f32_wide_batches(dtype, d, n_kv, group, batch, bad):
    """The step with batches on both sides of the 256 sequences one wave scans
    and of the 4096 of a launch, and one whose partial rows fill the workspace's
    bound; sequence `bad` is longer than its table: nothing is appended for it,
    and it is counted."""
    ctx = [(7 * i) % 61 for i in range(batch)]
    cfg = workloads.Config("wide", n_kv * group, n_kv, d, 16, dtype, batch)
    w, pa, pb, host, tables, lens, k_new, v_new = _setup(cfg, ctx, seed=21 + batch)
    lens[bad] = tables.shape[1] * 16 + 5
    mask = np.arange(batch) != bad
    q = np.random.default_rng(9).standard_normal((batch, n_kv * group, d)).astype(np.float32)
    q, got = _run_pair(cfg, pa, pb, host, tables, lens, k_new, v_new, q, q_f32=True, append_mask=mask)
    want = host.paged_decode(q[mask], tables[mask], lens[mask], chunk=64)
    assert rel_err(got[mask], want) <= TOL_F32
    assert pa.error_count() > 0 and pb.error_count() > 0


@pytest.mark.parametrize("d,n_kv,group,batch,width", [(256, 4, 4, 40, 130), (160, 8, 2, 300, 24), (224, 2, 20, 70, 160)])
def test_decode_f32_wide_heads_lone_waves(d, n_kv, group, batch, width):
    """bf16 queries over bf16 pages past 128 elements where the launch is wide
    enough (by its table) for a wave to a tile: the step's pages and outputs, and
    few splits."""
    ctx = [(37 * i) % 300 for i in range(batch)]
    cfg = workloads.Config("lone", n_kv * group, n_kv, d, 16, airkv.BF16, batch)
    w, pa, pb, host, tables, lens, k_new, v_new = _setup(cfg, ctx, seed=51 + d)
    tables = np.pad(tables, ((0, 0), (0, max(0, width - tables.shape[1]))), constant_values=-1)
    q = np.random.default_rng(11).standard_normal((batch, n_kv * group, d)).astype(np.float32)
    q, got = _run_pair(cfg, pa, pb, host, tables, lens, k_new, v_new, q, q_f32=False)
    want = host.paged_decode(q, tables, lens, chunk=64)
    err = rel_err(got, want)
    torch = torch_mod()
    qt, tt, lt = torch.from_numpy(q).cuda().to(torch.bfloat16), torch.from_numpy(tables).cuda(), torch.from_numpy(lens).cuda()
    for most in (1, 8):
        out = torch.full(q.shape, float("nan"), device="cuda")
        pb.paged_decode(qt, tt, lt, out, max_splits=most)
        err = max(err, rel_err(out.cpu().numpy(), want))
    log(f"decode f32 lone waves d={d}: rel err {err:.2e}")
    assert err <= TOL_F32


@pytest.mark.parametrize("dtype,d", [(airkv.BF16, 64), (airkv.INT8, 96), (airkv.F32, 224)])
def test_decode_f32_one_partition(dtype, d):
    """max_splits 1: a sequence's result does not depend on the others of its
    batch, bit for bit."""
    torch = torch_mod()
    lens = [0, 1, 16, 17, 33, 64, 65, 1000, 300, 2049]
    cfg = workloads.Config("one", 8, 2, d, 16, dtype, len(lens))
    _, _, (pool, host, tables, seq_lens, q, _) = _decode_case(cfg, lens, seed=5 + d)
    q, tables, seq_lens = (torch.from_numpy(x).cuda() for x in (q, tables, seq_lens))
    out, one = torch.full(q.shape, float("nan"), device="cuda"), torch.full(q.shape, float("nan"), device="cuda")
    pool.paged_decode(q, tables, seq_lens, out, max_splits=1)
    for i in range(len(lens)):
        pool.paged_decode(q[i:i + 1], tables[i:i + 1], seq_lens[i:i + 1], one[i:i + 1], max_splits=1)
    assert torch.equal(out, one) and bool(torch.isfinite(out).all())


@pytest.mark.parametrize("d,q_bf16", [(64, False), (96, False), (64, True), (96, True)])
def test_decode_f32_every_fp8_code(d, q_bf16):
    """Pages written as raw blocks may hold any code: subnormal ones, which the
    format reads as zero, and 0xFF, which it reads as -480 (0x7F, NaN, is left
    out), here in single tiles of a sequence; and an entry outside the pool is
    skipped and counted."""
    torch = torch_mod()
    n, bs, kv, group = 1000, 16, 2, 4
    cfg = workloads.Config("codes", kv * group, kv, d, bs, airkv.FP8, 1)
    w, pool, _, host, tables, lens, _, _ = _setup(cfg, [n - 1], seed=3)
    rng = np.random.default_rng(4)
    for x in (host.k, host.v):
        codes = np.arange(256, dtype=np.uint8)
        x[:] = rng.choice(codes[(codes != 0x7F) & (codes != 0xFF)], x.shape)
        for b in (3, 17):
            x[tables[0, b]] = rng.choice(codes[codes != 0x7F], x[tables[0, b]].shape)
            x[tables[0, b], 0, 5, 1] = 0xFF
    for s in (host.k_scales, host.v_scales):
        s[:] = rng.uniform(1e-4, 1e-3, s.shape).astype(np.float32)
    raw = [np.ascontiguousarray(x).reshape(pool.num_blocks, -1).view(np.uint8)
           for x in (host.k, host.v, host.k_scales, host.v_scales)]
    pool.write_blocks(np.arange(pool.num_blocks, dtype=np.int32), np.concatenate(raw, 1))
    lens = np.array([n], np.int32)
    qt = torch.from_numpy(rng.standard_normal((1, kv * group, d)).astype(np.float32)).cuda()
    qt = qt.to(torch.bfloat16) if q_bf16 else qt
    q = qt.float().cpu().numpy()
    out = torch.empty(q.shape, device="cuda")
    pool.paged_decode(qt, torch.from_numpy(tables).cuda(), torch.from_numpy(lens).cuda(), out)
    want = host.paged_decode(q, tables, lens, chunk=64)
    assert np.isfinite(want).all() and rel_err(out.cpu().numpy(), want) <= TOL_F32
    # the last block's entry outside the pool: as if the sequence ended before it
    assert pool.error_count(reset=True) == 0
    tables[0, n // bs] = pool.num_blocks + 3
    pool.paged_decode(qt, torch.from_numpy(tables).cuda(), torch.from_numpy(lens).cuda(), out)
    want = host.paged_decode(q, tables, np.array([n // bs * bs], np.int32), chunk=64)
    assert rel_err(out.cpu().numpy(), want) <= TOL_F32
    assert pool.error_count(reset=True) > 0


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("dtype", [airkv.F32, airkv.BF16])
@pytest.mark.parametrize("case", ["huge", "tiny", "tiny_k", "tiny_q"])
def test_decode_f32_value_ranges(dtype, d, case):
    """Values near the largest f32 (scores grow along the sequence, so a later
    tile's probabilities are the largest), values and keys near the least normal
    one (keys against queries as large), against 64 bits."""
    torch = torch_mod()
    n, kv, group = 400, 2, 2
    cfg = workloads.Config("range", kv * group, kv, d, 16, dtype, 1)
    w, pool, _, host, tables, lens, _, _ = _setup(cfg, [n - 1], seed=3)
    rng = np.random.default_rng(4)
    k, v = (rng.standard_normal((n, kv, d)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((1, kv * group, d)).astype(np.float32)
    if case == "huge":
        v = (v * np.float32(1e35) + np.float32(1e36)).astype(np.float32)
        k[:, :, 0] = np.arange(n)[:, None] / 16 * np.sqrt(d)        # one nat per tile
        q[:, :, 0] = 1.0
    elif case == "tiny":
        v *= np.float32(1e-36)
    elif case == "tiny_k":
        k, q = k * np.float32(1e-35), q * np.float32(1e35)
    else:
        k, q = k * np.float32(1e35), q * np.float32(1e-35)
    slots = (tables[0, np.arange(n) // 16].astype(np.int64) * 16 + np.arange(n) % 16)
    pool.append(torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), torch.from_numpy(slots).cuda())
    qt, lens = torch.from_numpy(q).cuda(), np.array([n], np.int32)
    if dtype == airkv.BF16:
        k, v = (torch.from_numpy(x).to(torch.bfloat16).float().numpy() for x in (k, v))
    s = np.einsum("gd,ngd->gn", q[0].astype(np.float64), np.repeat(k, group, 1).astype(np.float64)) / np.sqrt(d)
    p = np.exp(s - s.max(1, keepdims=True))
    want = np.einsum("gn,ngd->gd", p / p.sum(1, keepdims=True), np.repeat(v, group, 1).astype(np.float64))
    for most in (64, 1):
        out = torch.full(q.shape, float("nan"), device="cuda")
        pool.paged_decode(qt, torch.from_numpy(tables).cuda(), torch.from_numpy(lens).cuda(), out, max_splits=most)
        err = float(np.abs(out.cpu().numpy()[0].astype(np.float64) - want).max() / np.abs(want).max())
        log(f"decode f32 {case} dtype={dtype} d={d}: rel err {err:.2e}")
        assert err <= TOL_F32
