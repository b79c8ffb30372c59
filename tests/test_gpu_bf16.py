"""GPU parity of the BF16 flash-attention path (mx_flash_attn through the C ABI)
against the CPU oracle (double-precision restatement of the reference's
cpu_oracle, tests/attention_test.cu:64-98) and the reference's own gates."""
import numpy as np
import pytest
import torch

import oracle
from miroxen_amd import AttnParams, attn_reference, flash_attn
from miroxen_amd.attention import flash_attn_uses_mfma
from miroxen_amd.synth import CONFIGS, make_inputs
from tests.helpers import cosine, max_abs, query_rows, reference_gate

pytestmark = pytest.mark.gpu


def _bits(t: torch.Tensor) -> np.ndarray:
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _f32(t: torch.Tensor) -> np.ndarray:
    return t.float().cpu().numpy()


def _run(fn, q, k, v, p, out_rows, ostride, guard=16):
    """Run fn into a guard-banded output buffer (filled with 0xffff); return output
    rows [Sq, Hq*D] and the raw buffer for guard checks."""
    n = ostride * out_rows + 2 * guard
    buf = torch.full((n,), -1, dtype=torch.int16, device=q.device)
    o = buf[guard:guard + ostride * out_rows]
    fn(q, k, v, o, p)
    torch.cuda.synchronize()
    return o.view(torch.bfloat16).view(out_rows, ostride), buf


def _check_guards(buf, guard, Sq, ostride, row_elems, rows):
    raw = buf.cpu().numpy()
    assert np.all(raw[:guard] == -1) and np.all(raw[-guard:] == -1), "output guard was overwritten"
    if ostride > row_elems:
        body = raw[guard:-guard].reshape(Sq, ostride)
        assert np.all(body[rows, row_elems:] == -1), "output token padding was overwritten"


def _make(Sq, Skv, Hq, Hkv, D, pad, mag, seed, dev):
    qs = Hq * D + pad if pad else Hq * D
    ks = Hkv * D + pad + 2 if pad else Hkv * D
    os_ = Hq * D + pad + 4 if pad else Hq * D
    g = torch.Generator(device=dev); g.manual_seed(seed)
    q = (torch.randn(Sq, qs, generator=g, device=dev) * mag).to(torch.bfloat16)
    k = (torch.randn(Skv, ks, generator=g, device=dev) * mag).to(torch.bfloat16)
    v = (torch.randn(Skv, ks, generator=g, device=dev) * mag).to(torch.bfloat16)
    return q, k, v, qs, ks, os_


# Reference correctness suite (tests/attention_test.cu:211-227):
# Sq, Skv, Hq, Hkv, D, causal, q_offset, pad, magnitude, scale
CASES = [
    (1, 1, 1, 1, 64, 0, 0, 0, 1.0, 0.0), (1, 17, 4, 1, 72, 1, 0, 5, 3.0, 0.0),
    (17, 1, 3, 1, 128, 1, 2, 8, 2.0, 0.0), (17, 129, 4, 2, 64, 0, 0, 5, 2.0, 0.0),
    (129, 17, 8, 2, 72, 1, 5, 8, 3.0, 0.0), (129, 129, 4, 1, 128, 0, 0, 5, 3.0, 0.0),
    (1000, 1000, 2, 1, 64, 0, 0, 0, 1.0, 0.0), (1000, 1000, 2, 1, 72, 0, 0, 0, 3.0, 0.0),
    (1000, 1117, 4, 1, 128, 1, 117, 5, 2.0, 0.0), (16, 16, 32, 8, 128, 1, 0, 0, 1.0, 0.0),
    (129, 193, 64, 8, 128, 1, 64, 8, 3.0, 0.0), (2048, 2048, 32, 8, 128, 1, 0, 0, 1.0, 0.0),
    (4096, 4225, 32, 8, 128, 0, 0, 0, 2.0, 0.0), (16384, 18384, 32, 32, 128, 0, 0, 0, 1.0, 0.0),
    (4096, 4096, 32, 32, 128, 0, 0, 0, 1.0, 0.0), (65536, 65536, 32, 32, 128, 0, 0, 0, 1.0, 0.0),
    (1024, 1024, 8, 8, 64, 0, 0, 0, 1.0, 0.0), (16384, 16384, 8, 8, 72, 0, 0, 0, 1.0, 0.0),
    (17, 1000, 4, 1, 72, 0, 0, 6, 2.0, 0.25), (17, 129, 2, 1, 128, 1, 1000, 0, 3.0, 0.0),
    (129, 129, 2, 1, 128, 0, 0, 0, 2.0, -0.125), (17, 129, 2, 1, 128, 1, -17, 0, 2.0, 0.0),
    (129, 129, 2, 1, 72, 1, -17, 5, 3.0, 0.0), (17, 129, 4, 1, 64, 1, 2 ** 31 - 1, 0, 1.0, 0.0),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + f"_c{c[5]}o{c[6]}p{c[7]}")
def test_reference_suite(cuda, case):
    Sq, Skv, Hq, Hkv, D, causal, off, pad, mag, scale = case
    print(f"case {case}", flush=True)
    q, k, v, qs, ks, os_ = _make(Sq, Skv, Hq, Hkv, D, pad, mag, 1234 + Sq + Skv, cuda)
    p = AttnParams(Sq=Sq, Skv=Skv, Hq=Hq, Hkv=Hkv, D=D, scale=scale, causal=causal, q_offset=off,
                   q_stride=qs if pad else 0, kv_stride=ks if pad else 0, o_stride=os_ if pad else 0)
    # every case of the reference suite runs the MFMA kernel, the padded-stride (pad 5,
    # 6: not multiples of 8 elements) cases included
    assert flash_attn_uses_mfma(q, k, v, q, p)
    out, buf = _run(flash_attn, q, k, v, p, Sq, os_)
    rows = query_rows(Sq, Hq)
    got = _f32(out[rows, : Hq * D])
    if Sq < 65536:
        want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), Sq, Skv, Hq, Hkv, D, scale, causal, off,
                                    q_stride=qs, kv_stride=ks, rows=np.array(rows, np.int32))
        want = want.reshape(len(rows), Hq * D)
    else:  # 65536^2: the naive GPU reference on the sampled rows only, as the reference
        # test does (tests/attention_test.cu:150-161)
        qs_rows = q[rows, : Hq * D].contiguous()
        rp = AttnParams(Sq=len(rows), Skv=Skv, Hq=Hq, Hkv=Hkv, D=D, scale=scale, kv_stride=p.kv_stride)
        ref, _ = _run(attn_reference, qs_rows, k, v, rp, len(rows), Hq * D)
        want = _f32(ref[:, : Hq * D])
    ok, err, tol, rr = reference_gate(got, want)
    assert ok, f"flash/oracle mismatch max_abs={err} limit={tol} rel_rms={rr}"
    _check_guards(buf, 16, Sq, os_, Hq * D, rows)


def test_naive_reference_matches_oracle(cuda):
    """attn_reference (naive GPU kernel) against the oracle on a small masked GQA case."""
    Sq, Skv, Hq, Hkv, D = 33, 300, 4, 2, 128
    q, k, v, *_ = _make(Sq, Skv, Hq, Hkv, D, 0, 2.0, 77, cuda)
    mask = (torch.rand(Skv, generator=torch.Generator().manual_seed(3)) > 0.3).to(torch.uint8)
    p = AttnParams(Sq=Sq, Skv=Skv, Hq=Hq, Hkv=Hkv, D=D, kv_valid=mask.to(cuda))
    out, _ = _run(attn_reference, q, k, v, p, Sq, Hq * D)
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), Sq, Skv, Hq, Hkv, D, kv_valid=mask.numpy())
    assert reference_gate(_f32(out), want.reshape(Sq, -1))[0]


def _config_check(cfg_id, cuda, extra_rows=()):
    cfg = CONFIGS[cfg_id]
    print(f"config {cfg_id} {cfg.name}", flush=True)
    q, k, v, mask = make_inputs(cfg, seed=cfg_id, device=cuda)
    S, H, D = cfg.S, cfg.H, cfg.D
    p = AttnParams(Sq=S, Skv=S, Hq=H, Hkv=H, D=D, kv_valid=mask)
    o = torch.empty_like(q)
    flash_attn(q, k, v, o, p)
    torch.cuda.synchronize()
    rows = sorted(set(query_rows(S, H)) | set(extra_rows))
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), S, S, H, H, D,
                                kv_valid=None if mask is None else mask.cpu().numpy(),
                                rows=np.array(rows, np.int32))
    got = _f32(o[rows])
    # BASELINE tolerances for the BF16 kernel vs the FP32 CPU reference
    c, e = cosine(got, want), max_abs(got, want)
    print(f"config {cfg_id}: cosine={c:.7f} max_abs={e:.3g}", flush=True)
    assert c >= 0.9999 and e <= 2e-2
    assert reference_gate(got, want.reshape(got.shape))[0]
    return q, k, v, mask, o


def test_config1_full(cuda):
    """Config 1 (S=1088, H=24, no mask): every row against the FP32 oracle."""
    cfg = CONFIGS[1]
    q, k, v, _ = make_inputs(cfg, seed=1, device=cuda)
    p = AttnParams(Sq=cfg.S, Skv=cfg.S, Hq=cfg.H, Hkv=cfg.H, D=128)
    o = torch.empty_like(q)
    flash_attn(q, k, v, o, p)
    torch.cuda.synchronize()
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), cfg.S, cfg.S, cfg.H, cfg.H, 128)
    got = _f32(o)
    assert cosine(got, want) >= 0.9999 and max_abs(got, want) <= 2e-2


def test_config2_masked(cuda):
    _config_check(2, cuda, extra_rows=range(0, 4352, 97))


def test_config4_masked(cuda):
    _config_check(4, cuda)


def test_config5_video(cuda):
    _config_check(5, cuda)


def test_mask_equals_compacted_keys(cuda):
    """Size-independent invariant at config-2 size: masked attention == attention over
    the compacted valid keys."""
    cfg = CONFIGS[2]
    q, k, v, mask = make_inputs(cfg, seed=21, device=cuda)
    S, H = cfg.S, cfg.H
    o1 = torch.empty_like(q); o2 = torch.empty_like(q)
    flash_attn(q, k, v, o1, AttnParams(Sq=S, Skv=S, Hq=H, Hkv=H, D=128, kv_valid=mask))
    sel = mask.bool()
    kc, vc = k[sel].contiguous(), v[sel].contiguous()
    flash_attn(q, kc, vc, o2, AttnParams(Sq=S, Skv=int(sel.sum()), Hq=H, Hkv=H, D=128))
    torch.cuda.synchronize()
    assert max_abs(_f32(o1), _f32(o2)) <= 8e-3
    assert cosine(_f32(o1), _f32(o2)) > 0.99999


@pytest.mark.parametrize("Skv", [20000, 3000])
def test_mask_bitmap_paths(cuda, Skv):
    """The key-padding bitmaps are built from 16-byte loads when the mask is 16-byte
    aligned (two 1024-key chunks per wave up front, the rest after: Skv = 20000 needs 20
    chunks) and from byte loads otherwise: a random mask at an aligned and at an odd
    address gives bit-identical outputs, both against the oracle on sampled rows."""
    Sq, H, D = 256, 2, 128
    print(f"mask bitmaps Skv={Skv}", flush=True)
    q, k, v, *_ = _make(Sq, Skv, H, H, D, 0, 1.0, Skv, cuda)
    g = torch.Generator().manual_seed(Skv)
    mask = (torch.rand(Skv, generator=g) > 0.35).to(torch.uint8)
    mask[Skv - 70:] = 0  # a dead tail spanning a tile boundary
    base = torch.zeros(Skv + 64, dtype=torch.uint8, device=cuda)
    aligned, odd = base[:Skv], base[17:17 + Skv]
    aligned.copy_(mask.to(cuda))
    o1 = torch.empty_like(q)
    flash_attn(q, k, v, o1, AttnParams(Sq=Sq, Skv=Skv, Hq=H, Hkv=H, D=D, kv_valid=aligned))
    torch.cuda.synchronize()
    odd.copy_(mask.to(cuda))
    o2 = torch.empty_like(q)
    flash_attn(q, k, v, o2, AttnParams(Sq=Sq, Skv=Skv, Hq=H, Hkv=H, D=D, kv_valid=odd))
    torch.cuda.synchronize()
    assert odd.data_ptr() % 16 != 0 and aligned.data_ptr() % 16 == 0
    assert torch.equal(o1.view(torch.int16), o2.view(torch.int16))
    rows = np.array([0, 1, 100, 255], np.int32)
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), Sq, Skv, H, H, D, kv_valid=mask.numpy(), rows=rows)
    got = _f32(o1)[rows].reshape(want.shape)
    assert cosine(got, want) >= 0.9999 and max_abs(got, want) <= 2e-2


@pytest.mark.parametrize("Sq,H,Skv,D,causal", [
    (40, 2, 1, 128, 0), (40, 2, 3, 64, 0), (300, 24, 66, 128, 0), (300, 24, 67, 72, 0), (130, 24, 257, 128, 0),
    (500, 32, 1022, 128, 1), (300, 8, 1025, 128, 0), (256, 2, 2047, 64, 0), (256, 3, 17 * 1024 + 2, 128, 0),
])
def test_mask_of_a_partial_last_word(cuda, Sq, H, Skv, D, causal):
    """Masks of a length that is no multiple of four: the last keys count. Three of four
    keys are padding, so that each of the last ones weighs in the result; the 16-byte path
    and the byte path (odd mask address) give the same bits, whatever follows the mask."""
    print(f"partial last word Sq={Sq} H={H} Skv={Skv} D={D} causal={causal}", flush=True)
    q, k, v, *_ = _make(Sq, Skv, H, H, D, 0, 1.0, Skv, cuda)
    g = torch.Generator().manual_seed(Skv)
    mask = (torch.rand(Skv, generator=g) < 0.25).to(torch.uint8) * 3
    mask[Skv & ~3:] = 1
    outs = []
    for off in (0, 1):
        m = torch.full((Skv + 64,), 1, dtype=torch.uint8, device=cuda)
        m[off:off + Skv] = mask.to(cuda)
        p = AttnParams(Sq=Sq, Skv=Skv, Hq=H, Hkv=H, D=D, causal=causal, q_offset=Skv - Sq if causal else 0,
                       kv_valid=m[off:off + Skv])
        outs.append(_run(flash_attn, q, k, v, p, Sq, H * D)[0].clone())
    rows = sorted(set(range(0, Sq, max(1, Sq // 23))) | {Sq - 1})
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), Sq, Skv, H, H, D, 0.0, causal, Skv - Sq if causal else 0,
                                kv_valid=mask.numpy(), rows=np.array(rows, np.int32)).reshape(len(rows), -1)
    for o in outs:
        ok, err, tol, rr = reference_gate(_f32(o[rows]), want)
        assert ok, f"max_abs={err} limit={tol} rel_rms={rr}"
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


def test_all_masked_and_deterministic(cuda):
    S, H = 300, 2
    q, k, v, *_ = _make(S, S, H, H, 128, 0, 1.0, 5, cuda)
    zero = torch.zeros(S, dtype=torch.uint8, device=cuda)
    o = torch.full_like(q, 7.0)
    flash_attn(q, k, v, o, AttnParams(Sq=S, Skv=S, Hq=H, Hkv=H, D=128, kv_valid=zero))
    torch.cuda.synchronize()
    assert torch.all(o == 0)
    o1 = torch.empty_like(q); o2 = torch.empty_like(q)
    p = AttnParams(Sq=S, Skv=S, Hq=H, Hkv=H, D=128)
    flash_attn(q, k, v, o1, p); flash_attn(q, k, v, o2, p)
    torch.cuda.synchronize()
    assert torch.equal(o1.view(torch.int16), o2.view(torch.int16))


# Causal / q_offset / GQA on the MFMA path (D = 128, dense aligned strides): the
# reference's causal rule is key j visible to query row i iff j <= q_offset + i
# (attention.cu:108, :216-221); rows that see no key produce 0.
# Sq, Skv, Hq, Hkv, q_offset, masked
CAUSAL = [
    (1, 64, 1, 1, 0, False), (300, 300, 4, 4, 0, False), (1000, 1000, 4, 2, 0, False),
    (513, 1200, 2, 1, 687, False), (700, 700, 2, 2, -100, False), (700, 650, 2, 2, -300, False),
    (257, 2000, 2, 2, 2 ** 31 - 1, False), (4096, 4096, 8, 8, 0, False), (2048, 2300, 4, 4, 252, True),
]


@pytest.mark.parametrize("case", CAUSAL, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}x{c[3]}_o{c[4]}{'_m' if c[5] else ''}")
def test_causal_fast_path(cuda, case):
    Sq, Skv, Hq, Hkv, off, masked = case
    print(f"causal case {case}", flush=True)
    q, k, v, *_ = _make(Sq, Skv, Hq, Hkv, 128, 0, 1.0, 4321 + Sq + Skv, cuda)
    mask = None
    if masked:  # text-prefix style padding: 56 of the first 256 keys invalid
        m = torch.ones(Skv, dtype=torch.uint8)
        m[torch.randperm(256, generator=torch.Generator().manual_seed(5))[:56]] = 0
        mask = m
    p = AttnParams(Sq=Sq, Skv=Skv, Hq=Hq, Hkv=Hkv, D=128, causal=1, q_offset=off,
                   kv_valid=None if mask is None else mask.to(cuda))
    out, buf = _run(flash_attn, q, k, v, p, Sq, Hq * 128)
    rows = sorted(set(query_rows(Sq, Hq)) | set(range(0, Sq, max(1, Sq // 61))) | {Sq - 1})
    got = _f32(out[rows])
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), Sq, Skv, Hq, Hkv, 128, 0.0, 1, off,
                                kv_valid=None if mask is None else mask.numpy(),
                                rows=np.array(rows, np.int32)).reshape(len(rows), -1)
    # rows with no visible key are exactly 0
    dead = [i for i, r in enumerate(rows) if off + r < 0]
    if dead:
        assert np.all(got[dead] == 0)
    ok, err, tol, rr = reference_gate(got, want)
    assert ok, f"max_abs={err} limit={tol} rel_rms={rr}"
    live = [i for i, r in enumerate(rows) if off + r >= 0]
    assert cosine(got[live], want[live]) >= 0.9999 and max_abs(got, want) <= 2e-2
    _check_guards(buf, 16, Sq, Hq * 128, Hq * 128, rows)


def test_causal_equals_truncated_keys(cuda):
    """Size-independent invariant: row i of causal attention (q_offset = 0) equals
    non-causal attention of that row over keys 0..i."""
    S, H = 3000, 4
    q, k, v, *_ = _make(S, S, H, H, 128, 0, 1.0, 99, cuda)
    o = torch.empty_like(q)
    flash_attn(q, k, v, o, AttnParams(Sq=S, Skv=S, Hq=H, Hkv=H, D=128, causal=1))
    for i in (0, 63, 64, 255, 256, 1000, 2999):
        oi = torch.empty_like(q[i:i + 1])
        flash_attn(q[i:i + 1].contiguous(), k[: i + 1].contiguous(), v[: i + 1].contiguous(), oi,
                   AttnParams(Sq=1, Skv=i + 1, Hq=H, Hkv=H, D=128))
        torch.cuda.synchronize()
        assert max_abs(_f32(o[i:i + 1]), _f32(oi)) <= 4e-3, i


# D = 64 and D = 72 on the MFMA path, with NaN in the stride padding after each
# token's heads (D = 72 reads past the head in 16-byte chunks and must ignore it).
# Sq, Skv, Hq, Hkv, D, causal, q_offset, masked
SMALL_D = [
    (1000, 1000, 4, 2, 64, 0, 0, False), (1000, 1000, 4, 2, 72, 0, 0, False),
    (777, 1200, 6, 3, 72, 1, 423, False), (513, 513, 2, 2, 64, 1, 0, True),
    (2048, 2048, 8, 8, 72, 0, 0, True), (70, 4000, 3, 1, 72, 1, 3930, False),
]


@pytest.mark.parametrize("case", SMALL_D, ids=lambda c: "x".join(map(str, c[:5])) + f"_c{c[5]}o{c[6]}{'_m' if c[7] else ''}")
def test_small_head_dim_fast_path(cuda, case):
    Sq, Skv, Hq, Hkv, D, causal, off, masked = case
    print(f"small-D case {case}", flush=True)
    g = torch.Generator(device=cuda); g.manual_seed(777 + Sq + D)
    qs, ks = Hq * D + 8, Hkv * D + 8  # strides % 8 == 0: the fast path
    q = torch.randn(Sq, qs, generator=g, device=cuda).to(torch.bfloat16)
    k = torch.randn(Skv, ks, generator=g, device=cuda).to(torch.bfloat16)
    v = torch.randn(Skv, ks, generator=g, device=cuda).to(torch.bfloat16)
    for t, h in ((q, Hq), (k, Hkv), (v, Hkv)):
        t[:, h * D:] = float("nan")
    mask = None
    if masked:
        m = torch.ones(Skv, dtype=torch.uint8)
        m[torch.randperm(Skv, generator=torch.Generator().manual_seed(9))[: Skv // 5]] = 0
        mask = m
    p = AttnParams(Sq=Sq, Skv=Skv, Hq=Hq, Hkv=Hkv, D=D, causal=causal, q_offset=off, q_stride=qs, kv_stride=ks,
                   o_stride=Hq * D, kv_valid=None if mask is None else mask.to(cuda))
    out, buf = _run(flash_attn, q, k, v, p, Sq, Hq * D)
    rows = sorted(set(query_rows(Sq, Hq)) | set(range(0, Sq, max(1, Sq // 41))) | {Sq - 1})
    got = _f32(out[rows])
    assert np.all(np.isfinite(got))
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), Sq, Skv, Hq, Hkv, D, 0.0, causal, off,
                                q_stride=qs, kv_stride=ks, kv_valid=None if mask is None else mask.numpy(),
                                rows=np.array(rows, np.int32)).reshape(len(rows), -1)
    ok, err, tol, rr = reference_gate(got, want)
    assert ok, f"max_abs={err} limit={tol} rel_rms={rr}"
    assert cosine(got, want) >= 0.9999 and max_abs(got, want) <= 2e-2
    _check_guards(buf, 16, Sq, Hq * D, Hq * D, rows)


def test_d72_last_head_ends_the_allocation(cuda):
    """D = 72 reads 16-byte chunks past its 72 channels (to 80 of K, 96 of V). K and V here
    fill allocations of exactly 18 MiB (nine 2 MiB pages, no slack behind the last head of
    the last token), so a read past the last head would leave the mapping."""
    S, H, D = 8192, 16, 72
    assert S * H * D * 2 == 9 * 2 ** 21
    print(f"d72 allocation end S={S} H={H}", flush=True)
    q, k, v, *_ = _make(S, S, H, H, D, 0, 1.0, 72, cuda)
    p = AttnParams(Sq=64, Skv=S, Hq=H, Hkv=H, D=D)
    out, _ = _run(flash_attn, q, k, v, p, 64, H * D)
    rows = [0, 31, 63]
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), 64, S, H, H, D, 0.0, 0, 0,
                                rows=np.array(rows, np.int32)).reshape(len(rows), -1)
    assert reference_gate(_f32(out[rows]), want)[0]


# Grids of few units run 128-query units whose two wave groups take alternating key tiles and
# merge in LDS: numbers of key tiles odd and even, the last tile ragged, one group's keys
# all masked, rows that see no key, ragged query tiles, every head dim, padded and odd output
# strides (element-wise stores); and causal grids beyond one round of 256-query units, whose
# order over an XCD's heads differs for head counts that are no multiple of 8.
# Sq, Skv, Hq, Hkv, D, causal, q_offset, pad, dead keys [lo, hi)
KS = [
    (333, 333, 32, 8, 128, 1, 0, 0, (0, 0)), (129, 193, 24, 24, 128, 0, 0, 0, (0, 0)),
    (1, 257, 40, 8, 128, 1, 256, 0, (0, 0)), (300, 450, 16, 4, 128, 1, -70, 5, (0, 0)),
    (260, 320, 24, 24, 128, 0, 0, 0, (64, 128)), (200, 250, 24, 24, 128, 0, 0, 3, (128, 250)),
    (700, 1000, 16, 16, 72, 0, 0, 8, (0, 64)), (513, 300, 16, 8, 72, 1, 40, 6, (0, 0)),
    (385, 640, 24, 12, 64, 0, 0, 5, (0, 0)), (900, 1000, 8, 8, 64, 1, 100, 0, (300, 400)),
    (700, 700, 12, 12, 128, 1, 0, 0, (0, 0)),
    (2100, 2100, 32, 8, 128, 1, 0, 0, (0, 0)), (5600, 5600, 12, 4, 128, 1, 0, 0, (0, 0)),
    # behind a long cache: 256-query units again, one round of them
    (900, 3200, 48, 8, 128, 1, 2300, 0, (0, 0)), (1000, 3601, 64, 8, 72, 1, 2601, 5, (64, 128)),
]


@pytest.mark.parametrize("case", KS, ids=lambda c: "x".join(map(str, c[:5])) + f"_c{c[5]}o{c[6]}p{c[7]}")
def test_alternating_key_tiles(cuda, case):
    Sq, Skv, Hq, Hkv, D, causal, off, pad, dead = case
    print(f"alternating key tiles {case}", flush=True)
    q, k, v, qs, ks, os_ = _make(Sq, Skv, Hq, Hkv, D, pad, 1.5, 17 + Sq + D, cuda)
    mask = None
    if dead[1]:
        mask = torch.ones(Skv, dtype=torch.uint8)
        mask[dead[0]:dead[1]] = 0
    p = AttnParams(Sq=Sq, Skv=Skv, Hq=Hq, Hkv=Hkv, D=D, causal=causal, q_offset=off, q_stride=qs, kv_stride=ks,
                   o_stride=os_, kv_valid=None if mask is None else mask.to(cuda))
    out, buf = _run(flash_attn, q, k, v, p, Sq, os_)
    rows = sorted(set(query_rows(Sq, Hq)) | set(range(0, Sq, max(1, Sq // 29))) | {Sq - 1})
    got = _f32(out[rows, : Hq * D])
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), Sq, Skv, Hq, Hkv, D, 0.0, causal, off, q_stride=qs,
                                kv_stride=ks, kv_valid=None if mask is None else mask.numpy(),
                                rows=np.array(rows, np.int32)).reshape(len(rows), -1)
    ok, err, tol, rr = reference_gate(got, want)
    assert ok, f"max_abs={err} limit={tol} rel_rms={rr}"
    blind = [i for i, r in enumerate(rows) if causal and off + r < 0]
    assert np.all(got[blind] == 0)
    _check_guards(buf, 16, Sq, os_, Hq * D, rows)


# Key-range split of the grid's last round (flash_attn_split_plan): the split units'
# rows against the oracle, parts whose keys are all masked, GQA / D = 64 / 72 with
# padded strides, and repeat / cross-stream calls sharing the library's split region.
# Sq, Skv, Hq, Hkv, D, pad, dead_from (keys >= dead_from masked; 0: no mask)
SPLIT = [
    (1024, 1024, 2, 2, 128, 0, 700), (1000, 1000, 4, 2, 72, 5, 0), (600, 2000, 6, 3, 64, 8, 0),
    (4352, 4352, 6, 6, 128, 0, 4296), (257, 4000, 3, 1, 128, 0, 1000),
]


@pytest.mark.parametrize("case", SPLIT, ids=lambda c: "x".join(map(str, c[:5])) + f"_p{c[5]}d{c[6]}")
def test_split_grid(cuda, case):
    from miroxen_amd.attention import flash_attn_split_plan
    Sq, Skv, Hq, Hkv, D, pad, dead = case
    print(f"split case {case}", flush=True)
    q, k, v, qs, ks, os_ = _make(Sq, Skv, Hq, Hkv, D, pad, 1.0, 55 + Sq + D, cuda)
    mask = None
    if dead:
        mask = torch.ones(Skv, dtype=torch.uint8)
        mask[dead:] = 0
    p = AttnParams(Sq=Sq, Skv=Skv, Hq=Hq, Hkv=Hkv, D=D, q_stride=qs if pad else 0, kv_stride=ks if pad else 0,
                   o_stride=os_ if pad else 0, kv_valid=None if mask is None else mask.to(cuda))
    full, units, parts = flash_attn_split_plan(p)
    assert parts > 1 and units > 0, "case chosen to exercise the split"
    out, buf = _run(flash_attn, q, k, v, p, Sq, os_)
    # rows of split units: unit L = head * ntq + qtile, split units are L >= full
    ntq = (Sq + 255) // 256
    rows = sorted(set(query_rows(Sq, Hq)) | set(range(0, Sq, max(1, Sq // 53))) | {Sq - 1})
    got = _f32(out[rows, : Hq * D])
    want = oracle.attention_f64(_bits(q), _bits(k), _bits(v), Sq, Skv, Hq, Hkv, D, q_stride=qs, kv_stride=ks,
                                kv_valid=None if mask is None else mask.numpy(),
                                rows=np.array(rows, np.int32)).reshape(len(rows), -1)
    ok, err, tol, rr = reference_gate(got, want)
    assert ok, f"max_abs={err} limit={tol} rel_rms={rr}"
    assert cosine(got, want) >= 0.9999 and max_abs(got, want) <= 2e-2
    split_heads = sorted({L // ntq for L in range(full, full + units)})
    cols = np.concatenate([np.arange(h * D, (h + 1) * D) for h in split_heads])
    assert max_abs(got[:, cols], want[:, cols]) <= 2e-2
    _check_guards(buf, 16, Sq, os_, Hq * D, rows)
    # repeat: bit-identical
    out2, _ = _run(flash_attn, q, k, v, p, Sq, os_)
    assert torch.equal(out.view(torch.int16), out2.view(torch.int16))


def test_split_allocates_nothing(cuda):
    """A split call keeps its partials in the library's fixed device region: the free
    device memory is the same before and after the first split calls of three head
    dims (the region is part of the loaded code object, not allocated on the launch
    path), and the results still meet the BF16 gates."""
    from miroxen_amd.attention import flash_attn_split_plan
    warm = _make(256, 256, 1, 1, 128, 0, 1.0, 3, cuda)
    flash_attn(warm[0], warm[1], warm[2], torch.empty_like(warm[0]), AttnParams(Sq=256, Skv=256, Hq=1, Hkv=1, D=128))
    cases = []
    for D, seed in ((128, 31), (64, 32), (72, 33)):
        Sq, Skv, H = 512, 4096, 4
        q, k, v, *_ = _make(Sq, Skv, H, H, D, 0, 1.0, seed, cuda)
        p = AttnParams(Sq=Sq, Skv=Skv, Hq=H, Hkv=H, D=D)
        assert flash_attn_split_plan(p)[2] > 1, D
        cases.append((q, k, v, p, torch.empty_like(q), torch.empty_like(q)))
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    for q, k, v, p, o, _ in cases:
        flash_attn(q, k, v, o, p)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free0
    for q, k, v, p, o, ref in cases:
        attn_reference(q, k, v, ref, p)
        torch.cuda.synchronize()
        assert cosine(_f32(o), _f32(ref)) >= 0.9999 and max_abs(_f32(o), _f32(ref)) <= 2e-2, p.D


def test_split_calls_on_two_streams(cuda):
    """Two split calls on different streams share the library's partial region; the
    second waits for the first's merge, so both results equal their single-stream runs."""
    S, H = 1024, 4
    q1, k1, v1, *_ = _make(S, S, H, H, 128, 0, 1.0, 8, cuda)
    q2, k2, v2, *_ = _make(S, S, H, H, 128, 0, 2.0, 9, cuda)
    p = AttnParams(Sq=S, Skv=S, Hq=H, Hkv=H, D=128)
    ref1, ref2 = torch.empty_like(q1), torch.empty_like(q2)
    flash_attn(q1, k1, v1, ref1, p); flash_attn(q2, k2, v2, ref2, p)
    torch.cuda.synchronize()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    o1, o2 = torch.empty_like(q1), torch.empty_like(q2)
    for _ in range(3):
        with torch.cuda.stream(s1):
            flash_attn(q1, k1, v1, o1, p, stream=s1)
        with torch.cuda.stream(s2):
            flash_attn(q2, k2, v2, o2, p, stream=s2)
        torch.cuda.synchronize()
        assert torch.equal(o1.view(torch.int16), ref1.view(torch.int16))
        assert torch.equal(o2.view(torch.int16), ref2.view(torch.int16))


def test_graph_capture_replays(cuda):
    """flash_attn and flash_attn_fp8 captured into a HIP graph (torch.cuda.graph) and
    replayed with eager work in between: every replay equals the first bit for bit and
    the eager result to the BF16 tolerance. Under capture flash_attn does not split its
    grid (the library's split region is shared with eager calls, which a graph replay
    cannot be ordered against), so a captured replay differs from the eager result by
    rounding only."""
    from miroxen_amd import flash_attn_fp8, flash_attn_fp8_workspace
    from miroxen_amd.attention import flash_attn_split_plan
    S, H = 1024, 2
    q, k, v, *_ = _make(S, S, H, H, 128, 0, 1.0, 61, cuda)
    p = AttnParams(Sq=S, Skv=S, Hq=H, Hkv=H, D=128)
    assert flash_attn_split_plan(p)[2] > 1  # eager calls of this shape split
    eager, eager8 = torch.empty_like(q), torch.empty_like(q)
    ws = torch.zeros(flash_attn_fp8_workspace(p), dtype=torch.uint8, device=cuda)
    flash_attn(q, k, v, eager, p)
    flash_attn_fp8(q, k, v, eager8, p, ws)
    torch.cuda.synchronize()
    o, o8 = torch.empty_like(q), torch.empty_like(q)
    g = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # warm-up on the capture stream, as torch recommends
        flash_attn(q, k, v, o, p)
        flash_attn_fp8(q, k, v, o8, p, ws)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        flash_attn(q, k, v, o, p)
        flash_attn_fp8(q, k, v, o8, p, ws)
    outs = []
    for i in range(3):
        o.fill_(0); o8.fill_(0)
        g.replay()
        torch.cuda.synchronize()
        outs.append((o.clone(), o8.clone()))
        flash_attn(q, k, v, eager, p)  # eager work between replays (uses the split region)
        torch.cuda.synchronize()
    for a, b in outs[1:]:
        assert torch.equal(a.view(torch.int16), outs[0][0].view(torch.int16))
        assert torch.equal(b.view(torch.int16), outs[0][1].view(torch.int16))
    assert max_abs(_f32(outs[0][0]), _f32(eager)) <= 4e-3
    assert cosine(_f32(outs[0][0]), _f32(eager)) > 0.99999
    assert torch.equal(outs[0][1].view(torch.int16), eager8.view(torch.int16))
