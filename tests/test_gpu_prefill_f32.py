"""Prefill at f32 precision (f32 pages, head_dim other than 128) against the
oracle's blockwise attention, at the edges of its tiles: columns (query rows
times the GQA group) around a wave's 32 and a workgroup's 32 to 128, keys around
the 32- to 128-key tiles, head_dim below each built size, and launches whose
waves share a column set's keys four, two and one ways; and the row-by-row kernel
that small launches of these pools take, on each of its builds."""
import ctypes

import numpy as np
import pytest

import airkv
from airkv import workloads
from gpu_helpers import log, rel_err, torch_mod
from test_gpu_prefill import _prefill_case, _setup

pytestmark = pytest.mark.gpu

# Both sides sum in f32 in orders of their own: at most n * 2^-24 apart for n
# <= 840 keys (5e-5) relative to the largest output; twice that covers the
# scores' own rounding.
TOL_F32 = 1e-4


# (dtype, head_dim, kv heads, group, block size, query lengths, contexts)
CASES = [
    # few columns, long prefixes: four key shares (two from 97 elements on, one
    # for f32 / 1-byte pages past 128)
    (dt, d, 1, 8, 16, [1, 4, 5, 2], [701, 64 + 4, 840, 129]) for dt, d in
    [(airkv.BF16, 64), (airkv.BF16, 96), (airkv.BF16, 256), (airkv.F32, 64), (airkv.F32, 96), (airkv.F32, 128),
     (airkv.F32, 256), (airkv.INT8, 64), (airkv.FP8, 96), (airkv.INT8, 256)]
] + [
    # whole workgroups and one column more, no prefix and ragged ones
    (dt, d, 4, 4, 32, [31, 32, 33, 97, 128, 1, 200], [31, 32 + 31, 33 + 65, 97, 128 + 256, 300, 200]) for dt, d in
    [(airkv.BF16, 32), (airkv.BF16, 64), (airkv.BF16, 96), (airkv.BF16, 160), (airkv.BF16, 256), (airkv.F32, 64),
     (airkv.F32, 128), (airkv.F32, 224), (airkv.FP8, 64), (airkv.INT8, 96)]
] + [
    # columns that are no multiple of the group's rows, one head per kv head,
    # a group above the vector kernel's eight heads
    (airkv.BF16, 64, 8, 7, 16, [63, 64, 65, 130, 9, 300], [63, 64 + 1, 65 + 400, 130, 9 + 77, 300]),
    (airkv.F32, 64, 8, 1, 16, [255, 257, 129, 511, 1, 37], [255, 257 + 9, 129, 511, 1, 400]),
    (airkv.F32, 128, 2, 12, 16, [90, 170], [90, 170 + 33]),
]


@pytest.mark.parametrize("q_bf16", [True, False])
@pytest.mark.parametrize("dtype,d,n_kv,group,bs,q_lens,ctx", CASES)
def test_prefill_f32_tile_edges(dtype, d, n_kv, group, bs, q_lens, ctx, q_bf16):
    cfg = workloads.Config("f32", n_kv * group, n_kv, d, bs, dtype, len(ctx))
    got, want = _prefill_case(cfg, ctx, q_lens, seed=31 + d + group, q_bf16=q_bf16)
    err = rel_err(got, want)
    log(f"prefill f32 dtype={dtype} d={d} group={group} q_bf16={q_bf16}: rel err {err:.2e}")
    assert err <= TOL_F32


def _rule(dtype, d, n_kv, group, q_bf16, q_lens, tokens):
    """Whether such a launch takes the f32-precision kernel (else the row kernel)."""
    f = airkv.load().airkv_prefill_f32_better
    f.argtypes = [ctypes.c_int32] * 8 + [ctypes.c_int64]
    return f(dtype, d, n_kv, group, airkv.BF16 if q_bf16 else airkv.F32, sum(q_lens), len(q_lens), max(q_lens), tokens)


# (head_dim, kv heads, group): every width and head count the row kernel is built for
ROWS = [(32, 4, 1), (64, 2, 2), (64, 1, 4), (32, 1, 3), (96, 4, 1), (96, 2, 2), (96, 1, 4), (160, 4, 1), (256, 2, 2),
        (224, 1, 3), (192, 1, 8), (256, 1, 12)]


@pytest.mark.parametrize("dtype,d,n_kv,group,q_bf16",
                         [(dt, d, kv, g, qb) for dt in (airkv.F32, airkv.BF16, airkv.INT8, airkv.FP8) for d, kv, g in ROWS
                          for qb in (False, True) if not qb or (g == 1 and d != 32)] +
                         [(airkv.F32, 128, kv, g, False) for kv, g in ((4, 1), (2, 2), (1, 4))])
def test_prefill_rows_small_chunks(dtype, d, n_kv, group, q_bf16):
    """Chunks of 1 to 8 rows over 0 to 61 tokens before them: the row kernel."""
    q_lens, ctx = [8, 5, 1, 3], [40, 5, 64, 20]
    assert not _rule(dtype, d, n_kv, group, q_bf16, q_lens, 64)
    cfg = workloads.Config("rows", n_kv * group, n_kv, d, 16, dtype, len(ctx))
    got, want = _prefill_case(cfg, ctx, q_lens, seed=43 + d + group, q_bf16=q_bf16)
    assert rel_err(got, want) <= TOL_F32


@pytest.mark.parametrize("dtype,d", [(airkv.BF16, 64), (airkv.F32, 64), (airkv.F32, 128)])
def test_prefill_f32_non_finite_values_stay_behind_the_mask(dtype, d):
    """Non-finite elements of a value row reach the query rows that see that
    token, in their own channels; every other output is as with finite ones."""
    torch = torch_mod()
    n_kv, group, bs, n = 4, 4, 16, 200
    cfg = workloads.Config("inf", n_kv * group, n_kv, d, bs, dtype, 2)
    pool, host, tables, lens = _setup(cfg, [n, n], seed=5)
    at = 150                                             # token of sequence 0 that turns non-finite
    slot = np.array([tables[0, at // bs] * bs + at % bs], np.int64)
    k = np.random.default_rng(1).standard_normal((1, n_kv, d)).astype(np.float32)
    v = k.copy()
    v[0, :, [3, d - 1]] = 0.0
    host.append(k, v, slot)
    v[0, :, 3], v[0, :, d - 1] = np.inf, np.nan
    pool.append(torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), torch.from_numpy(slot).cuda())
    cu = np.array([0, n, 2 * n], np.int32)
    q = np.random.default_rng(2).standard_normal((2 * n, cfg.n_q_heads, d)).astype(np.float32)
    out = torch.empty(q.shape, device="cuda")
    pool.paged_prefill(torch.from_numpy(q).cuda(), torch.from_numpy(cu).cuda(), torch.from_numpy(tables).cuda(),
                       torch.from_numpy(lens).cuda(), out)
    torch.cuda.synchronize()
    got, want = out.cpu().numpy(), host.paged_prefill(q, cu, tables, lens)
    assert np.isposinf(got[at:n, :, 3]).all() and np.isnan(got[at:n, :, d - 1]).all()
    got[at:n, :, [3, d - 1]] = want[at:n, :, [3, d - 1]]
    assert np.isfinite(got).all()
    assert rel_err(got, want) <= TOL_F32


def test_prefill_f32_invalid_sequences():
    """A chunk longer than its sequence and a seq_len beyond the table are each
    counted once with their rows zero-filled; an out-of-pool table entry is
    counted once and read as zero keys and values; rows outside every sequence
    keep their bytes."""
    torch = torch_mod()
    cfg = workloads.Config("bad", 32, 8, 64, 16, airkv.BF16, 3)
    pool, host, tables, lens = _setup(cfg, [400, 300, 350], seed=79)
    q_lens = [200, 301, 100]
    lens_bad = lens.copy()
    lens_bad[2] = tables.shape[1] * 16 + 1
    cu = np.zeros(4, np.int32)
    cu[1:] = np.cumsum(q_lens)
    total = int(cu[-1])
    q = torch.randn((total + 3, 32, 64), device="cuda")
    out = torch.full((total + 3, 32, 64), 7.0, device="cuda")
    args = (torch.from_numpy(cu).cuda(), torch.from_numpy(tables).cuda())
    pool.error_count(reset=True)
    pool.paged_prefill(q, *args, torch.from_numpy(lens_bad).cuda(), out)
    torch.cuda.synchronize()
    assert pool.error_count(reset=True) == 2
    got = out.cpu().numpy()
    assert np.all(got[200:total] == 0.0) and np.all(got[total:] == 7.0)
    want = host.paged_prefill(q.cpu().numpy()[:200], cu[:2], tables[:1], lens[:1])
    assert rel_err(got[:200], want) <= TOL_F32
    # an out-of-pool entry: as a block of zeros
    t2 = tables.copy()
    t2[0, 3] = pool.num_blocks + 5
    hz = _host_with_zero_block(host, cfg)
    t3 = tables.copy()
    t3[0, 3] = host.num_blocks
    out.fill_(7.0)
    pool.paged_prefill(q, args[0], torch.from_numpy(t2).cuda(), torch.from_numpy(lens_bad).cuda(), out)
    torch.cuda.synchronize()
    assert pool.error_count(reset=True) == 3
    want = hz.paged_prefill(q.cpu().numpy()[:200], cu[:2], t3[:1], lens[:1])
    assert rel_err(out.cpu().numpy()[:200], want) <= TOL_F32


def _host_with_zero_block(host, cfg):
    import oracle
    hz = oracle.HostPool(host.num_blocks + 1, cfg.block_size, cfg.n_kv_heads, cfg.head_dim, cfg.dtype)
    hz.k[:host.num_blocks], hz.v[:host.num_blocks] = host.k, host.v
    return hz


@pytest.mark.parametrize("dtype,d", [(airkv.F32, 64), (airkv.F32, 128), (airkv.BF16, 64), (airkv.BF16, 256)])
@pytest.mark.parametrize("case", ["unit", "huge", "tiny", "tiny_channel", "tiny_k", "tiny_q", "spikes"])
def test_prefill_f32_value_ranges(dtype, d, case):
    """Values near the largest f32 and near 2^-106 (24 bits are kept from 2^-110 on),
    a channel of such among ordinary ones, keys of 1e-32 or 1e32 under queries of
    the opposite, and a few huge values, against 64 bits, channel by channel.  Sums
    of up to 300 f32 products in any order: within 300 * 2^-24 = 1.8e-5."""
    torch = torch_mod()
    n, kv, group = 300, 2, 4
    cfg = workloads.Config("range", kv * group, kv, d, 16, dtype, 2)
    pool, _, tables, lens = _setup(cfg, [n, n], seed=5)
    rng = np.random.default_rng(4)
    k, v = (rng.standard_normal((2 * n, kv, d)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((2 * n, kv * group, d)).astype(np.float32)
    if case == "huge":
        v *= np.float32(1e36)
    elif case == "tiny":
        v = ((np.abs(v) + 1) * np.float32(1e-32)).astype(np.float32)
    elif case == "tiny_channel":
        v[:, :, 5] = (np.abs(v[:, :, 5]) + 1) * np.float32(1e-32)
    elif case == "tiny_k":
        k, q = k * np.float32(1e-32), q * np.float32(1e32)
    elif case == "tiny_q":
        k, q = k * np.float32(1e32), q * np.float32(1e-32)
    elif case == "spikes":
        v.reshape(-1)[rng.integers(0, v.size, 5)] = 1e37
    slots = np.concatenate([t[np.arange(n) // 16].astype(np.int64) * 16 + np.arange(n) % 16 for t in tables])
    pool.append(torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), torch.from_numpy(slots).cuda())
    cu = np.array([0, n, 2 * n], np.int32)
    assert _rule(dtype, d, kv, group, False, [n, n], 304)
    out = torch.full(q.shape, float("nan"), device="cuda")
    pool.paged_prefill(torch.from_numpy(q).cuda(), torch.from_numpy(cu).cuda(), torch.from_numpy(tables).cuda(),
                       torch.from_numpy(lens).cuda(), out)
    got = out.cpu().numpy().astype(np.float64)
    if dtype == airkv.BF16:
        k, v = (torch.from_numpy(x).to(torch.bfloat16).float().numpy() for x in (k, v))
    want = np.empty_like(got)
    for b in range(2):
        r = slice(b * n, (b + 1) * n)
        for h in range(kv * group):
            s = q[r, h].astype(np.float64) @ k[r, h // group].astype(np.float64).T / np.sqrt(d)
            p = np.exp(np.where(np.tri(n, dtype=bool), s, -np.inf) - np.where(np.tri(n, dtype=bool), s, -np.inf).max(1, keepdims=True))
            want[r, h] = p / p.sum(1, keepdims=True) @ v[r, h // group].astype(np.float64)
    err = float((np.abs(got - want).max((0, 1)) / np.abs(want).max((0, 1))).max())
    log(f"prefill f32 {case} dtype={dtype} d={d}: worst channel's rel err {err:.2e}")
    assert err <= 1.8e-5
