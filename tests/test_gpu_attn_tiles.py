"""The fp32 matrix-core tile kernel (csrc/attn_tiles.hip) where it can go
wrong: row counts around its 16- and 32-row tiles, chunk and table-window
edges, every head dim and storage type, block sizes on both sides of its
16-token rule, dense and packed grids, split contexts, bad table entries, and
the row kernel that takes unaligned tensors.

Tolerances: fp32 rtol = atol = 1e-5 against the float64 oracle (outputs are
convex combinations of N(0, 1) values: |out| <= ~4, fp32 sums of <= 2^13 terms
err by < 1e-6 of that); bf16 / fp16 one rounding of such an output, 2^-8 * 4
and 2^-11 * 4."""
import numpy as np
import pytest
import torch

from oracle import paged_ref as ref
from serving import _native
from serving.fake_paged_attn import paged_attn_fwd, paged_mqa_decode

pytestmark = pytest.mark.gpu
DEV = "cuda"
ATOL = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -6, torch.float16: 2.0 ** -9}


def np64(t):
    return t.float().cpu().numpy().astype(np.float64)


def problem(q_lens, pasts, hq, hkv, d, bs, dtype, seed=0):
    rng = np.random.default_rng(seed)
    ends = [p + n for p, n in zip(pasts, q_lens)]
    nblk = [-(-e // bs) for e in ends]
    nb = sum(nblk) + 3
    perm = rng.permutation(np.arange(1, nb))
    table = np.zeros((len(ends), max(max(nblk), 1)), dtype=np.int32)
    at = 0
    for i, n in enumerate(nblk):
        table[i, :n] = perm[at:at + n]
        at += n
    g = torch.Generator(device=DEV).manual_seed(seed)
    mk = lambda *s: torch.randn(s, generator=g, device=DEV).to(dtype)  # noqa: E731
    qsl = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    return dict(q=mk(int(qsl[-1]), hq, d), k=mk(nb, bs, hkv, d), v=mk(nb, bs, hkv, d),
                table=torch.from_numpy(table).to(DEV),
                lens=torch.tensor(ends, dtype=torch.int32, device=DEV),
                qsl=torch.from_numpy(qsl).to(DEV), max_q=max(q_lens))


def check(p, dtype, causal=True):
    out, lse = paged_attn_fwd(p["q"], p["k"], p["v"], p["table"], p["lens"], p["qsl"], p["max_q"],
                              causal=causal)
    want, wl = ref.paged_attention(np64(p["q"]), np64(p["k"]), np64(p["v"]),
                                   p["table"].cpu().numpy(), p["lens"].cpu().numpy(),
                                   p["qsl"].cpu().numpy(), causal=causal)
    atol = ATOL[dtype]
    np.testing.assert_allclose(np64(out), want, rtol=1e-5 if dtype == torch.float32 else 0,
                               atol=atol)
    fin = np.isfinite(wl)
    got = lse.cpu().numpy().astype(np.float64)
    assert np.array_equal(np.isfinite(got), fin)
    np.testing.assert_allclose(got[fin], wl[fin], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,bs", [(8, 1, 64, 16), (4, 1, 32, 8), (8, 2, 128, 32),
                                         (3, 1, 64, 4), (12, 1, 32, 16), (10, 2, 128, 1)])
def test_row_and_chunk_edges(dtype, hq, hkv, d, bs):
    # query runs and contexts around 16/32-row tiles and 16/32-token chunks
    check(problem([1, 2, 4, 5, 17, 33], [0, 15, 12, 60, 47, 31], hq, hkv, d, bs, dtype), dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
def test_many_tiles(dtype, causal):
    # above 256 and 512 tiles of 32 rows: both sides of the launch shapes
    for q_lens in ([300, 290, 280, 260], [500, 490, 480, 470, 460]):
        check(problem(q_lens, [0] * len(q_lens), 8, 1, 64, 16, dtype), dtype, causal)


@pytest.mark.parametrize("bs", [8, 16])
def test_table_windows_and_split(bs):
    # contexts split over workgroups in 512-token partitions, each inside one
    # table window (255 blocks)
    check(problem([3, 1], [4200, 2037], 8, 1, 64, bs, torch.float32), torch.float32)


@pytest.mark.parametrize("hq,d,bs,ctx", [(8, 32, 16, 4200), (8, 64, 8, 2100), (3, 128, 8, 4100),
                                         (8, 64, 4, 1100), (5, 32, 2, 1100), (8, 64, 1, 700),
                                         (8, 32, 1, 270), (8, 128, 2, 511)])
@pytest.mark.parametrize("causal", [True, False])
def test_partition_across_table_windows(hq, d, bs, ctx, causal):
    # one workgroup's keys cross the end of a window of 255 blocks, once to
    # three times: every key counts once
    p = problem([4, 21], [ctx - 4, ctx - 37], hq, 1, d, bs, torch.float32)
    out = torch.empty_like(p["q"])
    lse = torch.empty(out.shape[:2], device=DEV)
    rc = _native.lib().pkv_paged_attention(
        out.data_ptr(), lse.data_ptr(), p["q"].data_ptr(), p["k"].data_ptr(), p["v"].data_ptr(),
        p["k"].shape[0], bs, p["table"].data_ptr(), p["table"].shape[1], p["lens"].data_ptr(),
        p["qsl"].data_ptr(), 2, 25, 21, 0, hq, 1, d, 0.0, int(causal), 8192, 0, None, 0, None,
        _native.stream_ptr(p["q"].device))
    _native.check(rc, "pkv_paged_attention")
    want, wl = ref.paged_attention(np64(p["q"]), np64(p["k"]), np64(p["v"]),
                                   p["table"].cpu().numpy(), p["lens"].cpu().numpy(),
                                   p["qsl"].cpu().numpy(), causal=causal)
    np.testing.assert_allclose(np64(out), want, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(lse.cpu().numpy(), wl, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_long_prompt_of_small_blocks(dtype):
    # one prompt with enough tiles for a single partition, past a window's end:
    # its last rows against the oracle (their queries alone see the same keys)
    n, last = 2100, 70
    p = problem([n], [0], 8, 1, 64, 8, dtype)
    out, lse = paged_attn_fwd(p["q"], p["k"], p["v"], p["table"], p["lens"], p["qsl"], n)
    want, wl = ref.paged_attention(np64(p["q"])[n - last:], np64(p["k"]), np64(p["v"]),
                                   p["table"].cpu().numpy(), p["lens"].cpu().numpy(),
                                   np.array([0, last], dtype=np.int32))
    np.testing.assert_allclose(np64(out)[n - last:], want, atol=ATOL[dtype],
                               rtol=1e-5 if dtype == torch.float32 else 0)
    np.testing.assert_allclose(lse.cpu().numpy()[n - last:], wl, rtol=1e-5, atol=1e-5)


def test_packed_grid():
    # one prompt among many decode rows, sequences past one scan block (256)
    rng = np.random.default_rng(1)
    pasts = [int(x) for x in rng.integers(0, 90, size=300)]
    q_lens = [1] * 300
    q_lens[137], q_lens[299] = 70, 33
    check(problem(q_lens, pasts, 8, 1, 64, 16, torch.float32), torch.float32)


def test_bounds_past_the_librarys_int():
    p = problem([1] * 5, [3, 70, 600, 900, 12], 8, 1, 64, 16, torch.float32)
    args = (p["q"], p["k"], p["v"], p["table"], p["lens"])
    want = paged_mqa_decode(*args)
    assert torch.equal(paged_mqa_decode(*args, max_kv_len=1 << 40), want)
    out = paged_mqa_decode(*args, max_kv_len=(1 << 32) + 5, part_tokens=1 << 40)
    torch.testing.assert_close(out, want, rtol=1e-5, atol=1e-5)


def test_no_visible_key_and_empty_runs():
    p = problem([2, 3, 4], [10, 20, 30], 8, 1, 64, 16, torch.float32)
    p["lens"][1] = 0
    p["qsl"] = torch.tensor([0, 2, 5, 5], dtype=torch.int32, device=DEV)
    p["q"] = p["q"][:5].contiguous()
    check(p, torch.float32)


@pytest.mark.parametrize("bs", [8, 16])
def test_bad_block_reads_zeros(bs):
    p = problem([20], [50], 8, 1, 64, bs, torch.float32)
    nb = p["k"].shape[0]
    k, v = p["k"].clone(), p["v"].clone()
    bad = int(p["table"][0, 1])
    p["table"][0, 1] = nb + 5
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    out = torch.empty_like(p["q"])
    rc = _native.lib().pkv_paged_attention(
        out.data_ptr(), None, p["q"].data_ptr(), p["k"].data_ptr(), p["v"].data_ptr(), nb, bs,
        p["table"].data_ptr(), p["table"].shape[1], p["lens"].data_ptr(), p["qsl"].data_ptr(), 1,
        20, 20, 0, 8, 1, 64, 0.0, 1, 0, 0, None, 0, status.data_ptr(),
        _native.stream_ptr(p["q"].device))
    _native.check(rc, "pkv_paged_attention")
    assert int(status.item()) == _native.PKV_STATUS_BAD_BLOCK
    k[bad] = 0
    v[bad] = 0
    p["table"][0, 1] = bad
    want, _ = ref.paged_attention(np64(p["q"]), np64(k), np64(v), p["table"].cpu().numpy(),
                                  p["lens"].cpu().numpy(), p["qsl"].cpu().numpy())
    np.testing.assert_allclose(np64(out), want, rtol=1e-5, atol=1e-5)


def test_unaligned_tensors_take_the_row_kernel():
    p = problem([5, 40], [30, 3], 8, 1, 64, 16, torch.float32)
    q = torch.empty(p["q"].numel() + 1, device=DEV)[1:].view(p["q"].shape)
    q.copy_(p["q"])
    assert q.data_ptr() % 16 != 0
    p["q"] = q
    check(p, torch.float32)


@pytest.mark.parametrize("q_lens,pasts", [([500], [0]), ([8, 8], [2000, 1500]), ([1, 40], [900, 3])])
@pytest.mark.parametrize("workspace", [True, False])
def test_unaligned_tensors_split(q_lens, pasts, workspace):
    # the row kernel in its own partitions, and unsplit where no workspace is given
    p = problem(q_lens, pasts, 8, 1, 64, 16, torch.float32)
    q = torch.empty(p["q"].numel() + 1, device=DEV)[1:].view(p["q"].shape)
    q.copy_(p["q"])
    out = torch.empty_like(p["q"])
    L, n, mk = _native.lib(), len(q_lens), max(a + b for a, b in zip(q_lens, pasts))
    if not workspace:
        mk = min(mk, 512)  # the tile rule's one piece; longer contexts grow it
    wsb = L.pkv_attention_workspace_bytes(n, p["max_q"], 8, 1, 64, p["table"].shape[1], 16, mk, 0,
                                          0)
    ws = torch.zeros(wsb, dtype=torch.uint8, device=DEV) if workspace else None
    assert wsb > 0
    rc = L.pkv_paged_attention(
        out.data_ptr(), None, q.data_ptr(), p["k"].data_ptr(), p["v"].data_ptr(),
        p["k"].shape[0], 16, p["table"].data_ptr(), p["table"].shape[1], p["lens"].data_ptr(),
        p["qsl"].data_ptr(), n, q.shape[0], p["max_q"], mk, 8, 1, 64, 0.0, 1, 0, 0,
        _native.ptr(ws), wsb if workspace else 0, None, _native.stream_ptr(q.device))
    _native.check(rc, "pkv_paged_attention")
    want, _ = ref.paged_attention(np64(p["q"]), np64(p["k"]), np64(p["v"]),
                                  p["table"].cpu().numpy(), p["lens"].cpu().numpy(),
                                  p["qsl"].cpu().numpy())
    np.testing.assert_allclose(np64(out), want, rtol=1e-5, atol=1e-5)
