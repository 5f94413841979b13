"""GPU parity of the decode-step kernels around the GEMVs (decode attention, greedy argmax,
embedding gather), through the C-ABI, against the CPU oracle on the same seeded inputs.

Mirrors the reference's tests/test_kernels.py test_decode_attn (335-345: D 64/128, GQA groups 1..8,
context lengths 1..4000 in one batch, max_seq 4096, tolerance 2e-3 + 1e-2 |ref|),
test_decode_work_reuse (348-355: one zeroed work buffer shared by launches of B = 8, 1, 4, 16, 2)
and test_argmax (208-221). Adds: a captured graph replayed while the context grows (the split
count is derived on the device), and the exact embedding gather.
"""
import numpy as np
import pytest

from tests._util import check, cuda, gpu, host, rng

pytestmark = gpu


@pytest.fixture(scope="module")
def hi():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from hipinfer_amd import hipinfer
    return hipinfer


@pytest.fixture(scope="module")
def O():
    from oracle import oracle
    return oracle


def attn_case(hi, O, lens, Hq, Hkv, D, S, seed, work=None):
    r = rng(seed)
    B = len(lens)
    q = (r.standard_normal((B, Hq * D))).astype(np.float16)
    kc = (r.standard_normal((B, Hkv, S, D))).astype(np.float16)
    vc = (r.standard_normal((B, Hkv, S, D))).astype(np.float16)
    pos = np.array([l - 1 for l in lens], np.int32)
    got = host(hi.decode_attn(cuda(q), cuda(kc), cuda(vc), cuda(pos), Hq, Hkv, work=work))
    ref = O.decode_attn(q, kc, vc, pos, Hq, Hkv)
    return got, ref


CASES = [[1], [37], [4000], [1, 300, 1024, 2049], list(range(5, 4000, 250))]
GROUPS = [(64, 8), (64, 4), (64, 1), (128, 4), (128, 3), (128, 1), (128, 7), (64, 7), (128, 8), (64, 2), (128, 6),
          (64, 5)]


@pytest.mark.parametrize("D,G", GROUPS, ids=[f"D{d}-G{g}" for d, g in GROUPS])
def test_decode_attn(hi, O, D, G):
    Hkv = 4 if G != 1 else 16
    for i, lens in enumerate(CASES):
        got, ref = attn_case(hi, O, lens, Hkv * G, Hkv, D, 4096, 500 + 10 * D + G + i)
        check(f"decode attn D={D} G={G} lens={lens if len(lens) <= 4 else f'{lens[0]}..{lens[-1]}'}", got, ref,
              2e-3, 1e-2)


def test_decode_attn_batch64(hi, O):
    """The batched decode step's shape (Llama-3.1-8B: Hkv 8, G 4, D 128) at 64 sequences and about
    1024 positions: one split per (sequence, kv head), so each wave runs four tiles in turn with the
    next tile's K and V in flight during the current one; ragged lengths end tiles part-way."""
    lens = [1024 - 13 * i for i in range(64)]
    got, ref = attn_case(hi, O, lens, 32, 8, 128, 1040, 650)
    check("decode attn B=64 lens=1024..205", got, ref, 2e-3, 1e-2)


@pytest.mark.parametrize("D,Hkv,G", [(64, 8, 8), (128, 8, 4), (128, 2, 5)], ids=["D64-G8", "D128-G4", "D128-G5"])
@pytest.mark.parametrize("B", [1, 3, 24, 70], ids=lambda b: f"B{b}")
def test_decode_attn_tile_and_split_edges(hi, O, D, Hkv, G, B):
    """Lengths at the edges of a wave's 32 keys, of 128 and 256 keys (a pass of a block of 4 and of 8 waves where one
    split runs) and of the split rule's steps up to 16 splits, at batches of both block widths, with
    infinities and NaN in the cache behind every length: keys past it must not take part. Runs of several
    tiles a wave and more than 16 splits: test_decode_attn_long_contexts."""
    edges = [1, 31, 32, 33, 127, 128, 129, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 2079, 2080]
    S, Hq = 2080, Hkv * G
    for first in range(len(edges) if B == 1 else 1):
        lens = [edges[(first + 5 * b) % len(edges)] for b in range(B)]
        r = rng(640 + B + first)
        q = r.standard_normal((B, Hq * D)).astype(np.float16)
        kc = np.empty((B, Hkv, S, D), np.float16)
        vc = np.empty((B, Hkv, S, D), np.float16)
        kc[:] = r.standard_normal((1, Hkv, S, D))
        vc[:] = r.standard_normal((1, Hkv, S, D))
        for b, n in enumerate(lens):
            kc[b, :, n:] = np.inf
            vc[b, :, n:] = np.nan
        pos = np.array(lens, np.int32) - 1
        got = host(hi.decode_attn(cuda(q), cuda(kc), cuda(vc), cuda(pos), Hq, Hkv))
        check(f"decode attn D={D} G={G} B={B} lens={lens[:4]}", got, O.decode_attn(q, kc, vc, pos, Hq, Hkv), 2e-3, 1e-2)


@pytest.mark.parametrize("D,Hkv,G", [(64, 8, 4), (128, 8, 4), (128, 2, 6)], ids=["D64-G4", "D128-G4", "D128-Hkv2"])
@pytest.mark.parametrize("lens", [[4097], [6000], [8500], [4096, 4097, 4352, 6000], [6100, 33, 2500]],
                         ids=lambda l: "-".join(map(str, l)))
def test_decode_attn_long_contexts(hi, O, D, Hkv, G, lens):
    """Blocks of 8 waves whose waves run several tiles (splits of over 256 keys), and merges of more than the 16
    splits that one round requests (17 to 34 at batch 1), with infinities and NaN in the cache behind every
    length."""
    r = rng(670 + len(lens) + lens[0] + D)
    B, S, Hq = len(lens), max(lens) + 32, Hkv * G
    q = r.standard_normal((B, Hq * D)).astype(np.float16)
    kc = r.standard_normal((B, Hkv, S, D)).astype(np.float16)
    vc = r.standard_normal((B, Hkv, S, D)).astype(np.float16)
    for b, n in enumerate(lens):
        kc[b, :, n:] = np.inf
        vc[b, :, n:] = np.nan
    pos = np.array(lens, np.int32) - 1
    got = host(hi.decode_attn(cuda(q), cuda(kc), cuda(vc), cuda(pos), Hq, Hkv))
    check(f"decode attn D={D} G={G} lens={lens}", got, O.decode_attn(q, kc, vc, pos, Hq, Hkv), 2e-3, 1e-2)


@pytest.mark.parametrize("D,Hkv,G", [(64, 4, 8), (128, 8, 4)], ids=["D64-G8", "D128-G4"])
@pytest.mark.parametrize("B,n", [(1, 64), (1, 700), (3, 300), (70, 200)])
def test_decode_attn_minus_infinite_logits(hi, D, Hkv, G, B, n):
    """Keys whose logit is -inf have weight 0, also where they are every key a wave sees first (its first 32,
    or its last, partly filled tile): the result is that of the other keys, in float64 on the CPU."""
    r = rng(680 + B + n)
    Hq = Hkv * G
    q = r.standard_normal((B, Hq * D)).astype(np.float16)
    q.reshape(B, Hq, D)[:, :, 5] = 1.0 + r.random((B, Hq))
    kc = r.standard_normal((B, Hkv, n, D)).astype(np.float16)
    vc = r.standard_normal((B, Hkv, n, D)).astype(np.float16)
    pos = np.full(B, n - 1, np.int32)
    for lo, hi_ in ((0, 32), (n - n % 32 if n % 32 else n - 32, n), (17, 60)):
        kb = kc.copy()
        kb[:, :, lo:hi_, 5] = -np.inf
        got = host(hi.decode_attn(cuda(q), cuda(kb), cuda(vc), cuda(pos), Hq, Hkv))
        keep = np.r_[0:lo, hi_:n]
        s = np.einsum("bhgd,bhkd->bhgk", q.reshape(B, Hkv, G, D).astype(np.float64), kc[:, :, keep].astype(np.float64))
        p = np.exp(s / np.sqrt(D) - (s / np.sqrt(D)).max(-1, keepdims=True))
        ref = np.einsum("bhgk,bhkd->bhgd", p, vc[:, :, keep].astype(np.float64)) / p.sum(-1)[..., None]
        check(f"decode attn D={D} B={B} n={n} keys {lo}..{hi_} at -inf", got, ref.reshape(B, Hq * D), 2e-3, 1e-2)


def splits_run(hi, B, Hkv, n, D=64):
    """Splits per (sequence, kv head) pair that a batch of B sequences of n keys ran, counted in the partial
    results left in the work buffer (none for one split); the output is checked on the way."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    kc, vc = (torch.randn(B, Hkv, n, D, device="cuda", generator=g).half() for _ in range(2))
    q = torch.randn(B, Hkv * D, device="cuda", generator=g).half()
    pos = torch.full((B,), n - 1, dtype=torch.int32, device="cuda")
    work = torch.zeros(hi.lib.hi_decode_work_bytes(B, Hkv, Hkv, D), dtype=torch.uint8, device="cuda")
    got = hi.decode_attn(q, kc, vc, pos, Hkv, Hkv, work=work).float().view(B, Hkv, D)
    s = (kc.float() * q.float().view(B, Hkv, 1, D)).sum(-1) / D ** 0.5
    ref = (torch.softmax(s, -1)[..., None] * vc.float()).sum(2)
    check(f"decode attn {B} x {n}", host(got), host(ref), 2e-3, 1e-2)
    sums = work[4096 * 4:].view(torch.float32).view(B, Hkv, 64, D + 2)[..., D + 1]
    count = (sums != 0).sum(-1)
    assert (count == count[0, 0]).all()
    return max(1, int(count[0, 0]))


@pytest.mark.parametrize("B,Hkv,n,splits", [
    (512, 1, 1024, 1), (512, 1, 1025, 1), (512, 1, 1900, 1), (64, 8, 1025, 1), (64, 8, 1900, 1),
    (44, 8, 2048, 2), (44, 8, 2049, 2), (44, 8, 2900, 2), (24, 8, 3072, 3), (24, 8, 3073, 4)])
def test_decode_attn_splits_of_long_uniform_batches(hi, B, Hkv, n, splits):
    """Pairs that alone give every CU two blocks stay one split at every length (a second would be a part-filled
    second round of blocks: the time of 64 x 1025 keys went up by a tenth over 64 x 1024), and 44 x 8 stay
    two; 24 x 8 take a fourth over 3072 keys. On 256 CUs."""
    if hi.lib.hi_device_cus() != 256:
        pytest.skip("the counts are those of 256 CUs")
    assert splits_run(hi, B, Hkv, n) == splits


@pytest.mark.parametrize("B", [1, 5, 24])
def test_decode_attn_one_split_up_to_256_keys(hi, B):
    """A short context needs no merge: two splits of 100 keys took a quarter longer than one of 200."""
    assert [splits_run(hi, B, 8, n) for n in (1, 129, 200, 256)] == [1] * 4
    assert splits_run(hi, B, 8, 257) > 1


@pytest.mark.parametrize("B,n,splits", [(1, 8192, 32), (1, 8193, 32), (1, 12000, 32), (2, 6000, 16), (3, 4000, 10),
                                        (4, 2000, 8), (4, 20000, 8)])
def test_decode_attn_8_wave_launch_has_one_block_per_cu(hi, B, n, splits):
    """Launches of 8-wave blocks, of which a CU holds one: no more of them than CUs, at any length (8 kv heads;
    on 256 CUs)."""
    if hi.lib.hi_device_cus() != 256:
        pytest.skip("the counts are those of 256 CUs")
    assert splits_run(hi, B, 8, n) == splits


def test_decode_work_reuse(hi, O):
    """One zeroed work buffer for launches of decreasing and increasing batch: the split counters
    must be left zeroed and never land in a larger launch's partials. One kv head per sequence
    means many splits per launch."""
    import torch
    D, Hkv, G = 128, 1, 4
    work = torch.zeros(hi.lib.hi_decode_work_bytes(16, Hkv * G, Hkv, D), dtype=torch.uint8, device="cuda")
    for B in [8, 1, 4, 16, 2]:
        got, ref = attn_case(hi, O, [2000 - 97 * b for b in range(B)], Hkv * G, Hkv, D, 2048, 600 + B, work=work)
        check(f"decode attn shared work B={B}", got, ref, 2e-3, 1e-2)
    assert int(work[:4096 * 4].view(torch.int32).abs().sum()) == 0, "split counters not left zeroed"


def test_decode_attn_graph_replay_growing_context(hi, O):
    """A captured launch stays valid as pos advances (the kernel reads pos on the device and picks
    its split count from it); every replay matches the oracle."""
    import torch
    r = rng(700)
    B, Hkv, G, D, S = 3, 8, 4, 128, 4096
    Hq = Hkv * G
    q = r.standard_normal((B, Hq * D)).astype(np.float16)
    kc = r.standard_normal((B, Hkv, S, D)).astype(np.float16)
    vc = r.standard_normal((B, Hkv, S, D)).astype(np.float16)
    qd, kd, vd = cuda(q), cuda(kc), cuda(vc)
    pos = torch.zeros(B, dtype=torch.int32, device="cuda")
    out = torch.empty(B, Hq * D, dtype=torch.float16, device="cuda")
    work = torch.zeros(hi.lib.hi_decode_work_bytes(B, Hq, Hkv, D), dtype=torch.uint8, device="cuda")
    hi.decode_attn(qd, kd, vd, pos, Hq, Hkv, out=out, work=work)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        hi.decode_attn(qd, kd, vd, pos, Hq, Hkv, out=out, work=work)
    for p in [[0, 5, 63], [64, 255, 256], [1000, 2047, 4095], [3, 700, 1500]]:
        pn = np.array(p, np.int32)
        pos.copy_(torch.from_numpy(pn))
        g.replay()
        torch.cuda.synchronize()
        check(f"decode attn graph replay pos={p}", host(out), O.decode_attn(q, kc, vc, pn, Hq, Hkv), 2e-3, 1e-2)


def test_argmax(hi, O):
    """The reference's cases (ties to the lowest index, NaN wins, all -inf and all NaN rows give 0,
    +inf), exact against the oracle, plus vocabulary-sized random rows and an odd V whose rows are
    not 16-byte aligned."""
    import torch
    r = rng(710)
    V = 32000
    lg = r.standard_normal((6, V)).astype(np.float16)
    lg[1, 100] = lg[1, 31999] = 20.0
    lg[2, 5000] = np.nan
    lg[2, 7] = np.nan
    lg[3] = -np.inf
    lg[4] = np.nan
    lg[5, 31999] = np.inf
    got = host(hi.argmax(cuda(lg)))
    assert np.array_equal(got, O.argmax(lg)), got
    for V in [128256, 151936, 32001, 7]:
        lg = r.standard_normal((5, V)).astype(np.float16)
        lg[0, V // 3] = lg[0, V - 1] = 30.0  # a tie far apart
        got = host(hi.argmax(cuda(lg)))
        assert np.array_equal(got, O.argmax(lg)), (V, got)
    assert host(hi.argmax(torch.zeros(0, 10, dtype=torch.float16, device="cuda"))).shape == (0,)


def test_embed(hi):
    r = rng(720)
    V, H = 1000, 2048
    table = r.standard_normal((V, H)).astype(np.float16)
    tok = np.array([0, 999, 17, 17, 500], np.int32)
    got = host(hi.embed(cuda(tok), cuda(table)))
    assert np.array_equal(got, table[tok])
