"""The four-wave GEMM (gemm_quad.hip): every tile shape its plan picks for the model's projections,
every compiled instance, ragged row counts around the tiles, and outputs that are only 8-byte
aligned.  (tests/test_quad_plan.py checks that the shapes here cover what the plan picks.)

An output's accumulation runs through K in order whatever the tile, so unsplit launches agree bit
for bit on the rows they share; the largest launch is held to an fp64 product."""

import pytest
import torch

from helpers import bf16_ulp, check_linear

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
SHAPES = {"qkv": (6144, 2560), "o": (2560, 4096), "gu": (9728, 2560), "down": (2560, 9728)}
# between them these counts take every tile shape that the plan picks for 257 to 16384 rows of these
# projections, with each epilogue that picks it; 257, 1025 and 2049 leave one row in the last row
# block, 1023 and 4095 fill all but one
ROWS = [257, 300, 399, 513, 601, 768, 800, 1023, 1025, 1200, 1500, 1600, 2049, 2600, 3000, 3100, 3300,
        4095, 4500, 6001]
# one launch of every compiled instance, ten K stages and more: (split, MT, NT) -> rows, outputs, K, for
# each epilogue that it is compiled for (split partials: one instance serves all)
INSTANCES = {
    ("split", 2, 2): (33, 128, 640), ("split", 2, 3): (33, 6144, 2560), ("split", 2, 4): (33, 4096, 9728),
    ("split", 2, 6): (33, 9728, 9728), ("split", 4, 3): (257, 128, 640), ("split", 4, 4): (385, 128, 9728),
    ("plain", 2, 2): (63, 4096, 640), ("plain", 2, 3): (33, 20480, 640), ("plain", 2, 4): (33, 30720, 640),
    ("plain", 2, 6): (33, 45056, 640), ("plain", 4, 3): (1025, 256, 640), ("plain", 4, 4): (257, 9728, 640),
    ("plain", 4, 5): (385, 9728, 640), ("plain", 4, 6): (8193, 512, 640), ("plain", 4, 8): (3073, 2560, 640),
    ("plain", 4, 10): (3073, 3072, 1152), ("plain", 6, 5): (8193, 640, 640),
    ("plain", 6, 6): (769, 9728, 1152), ("plain", 6, 8): (2817, 4096, 640), ("plain", 8, 4): (6913, 1024, 640),
    ("plain", 8, 5): (769, 9728, 640), ("plain", 8, 6): (3073, 3072, 640), ("plain", 8, 8): (4865, 2560, 640),
    ("swiglu", 2, 2): (33, 128, 640), ("swiglu", 2, 4): (33, 9728, 640), ("swiglu", 2, 6): (33, 20480, 640),
    ("swiglu", 4, 4): (257, 128, 640), ("swiglu", 4, 6): (257, 6144, 640), ("swiglu", 4, 8): (257, 9728, 640),
    ("swiglu", 4, 10): (385, 9728, 640), ("swiglu", 6, 6): (1537, 2560, 640),
    ("swiglu", 6, 8): (513, 9728, 640), ("swiglu", 8, 4): (641, 4096, 640), ("swiglu", 8, 6): (8193, 512, 640),
    ("swiglu", 8, 8): (577, 9728, 640),
}


@pytest.fixture(scope="module")
def ops():
    from qdecode import ops as o
    return o


def _operands(name, M):
    N, K = SHAPES[name]
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    r = lambda *s, std=1.0: torch.empty(s, dtype=BF, device="cuda").normal_(0, std, generator=g)  # noqa: E731
    return r(M, K), r(2 * N if name == "gu" else N, K, std=0.02), r(M, N, std=2.0)


def _linear(ops, name, x, w, res, **kw):
    epi = {"qkv": ops.EPI_NONE, "gu": ops.EPI_SWIGLU}.get(name, ops.EPI_RES)
    return ops.linear(x, w, epi, res=res[:x.shape[0]] if epi == ops.EPI_RES else None, **kw)


@pytest.mark.parametrize("name", list(SHAPES))
def test_every_tile_shape_agrees(ops, name):
    N, K = SHAPES[name]
    x, w, res = _operands(name, ROWS[-1])
    print(f"\n[case] {name}: {ROWS} rows", flush=True)
    full = _linear(ops, name, x, w, res)
    acc = x.double() @ w.double().t()
    if name == "gu":
        # first-order propagation of one ulp in bf16(gate), bf16(up) and bf16(silu), two of output
        gate, up = acc[:, :N].to(BF).float(), acc[:, N:].to(BF).float()
        sg = torch.sigmoid(gate)
        s = (gate * sg).to(BF).float()
        want = (s * up).to(BF)
        dsilu = (sg * (1 + gate * (1 - sg))).abs()
        bound = (up.abs() * (dsilu * bf16_ulp(gate) + bf16_ulp(s)) + s.abs() * bf16_ulp(up)
                 + 2 * bf16_ulp(torch.maximum(full.float().abs(), want.float().abs())) + 2 ** -12)
    elif name == "qkv":
        want = acc.to(BF)
        bound = 2 * bf16_ulp(torch.maximum(full.float().abs(), want.float().abs())) + 2 ** -9
    else:
        a = acc.to(BF).float()
        want = (res.float() + a).to(BF)
        bound = bf16_ulp(a) + 2 * bf16_ulp(torch.maximum(full.float().abs(), want.float().abs()))
    d = (full.float() - want.float()).abs()
    assert bool((d <= bound).all()), f"max excess {float((d - bound).max())}"
    for M in ROWS[:-1]:
        if name in ("o", "down") and M < 1024:
            continue                             # K is split: other sums (tested with the splits)
        part = _linear(ops, name, x[:M], w, res)
        assert torch.equal(part.view(torch.int16), full[:M].view(torch.int16)), f"{M} rows"


@pytest.mark.parametrize("name", ["o", "down"])
@pytest.mark.parametrize("M", [257, 384, 513, 1023])
def test_split_launches(ops, name, M):
    x, w, res = _operands(name, M)
    got = _linear(ops, name, x, w, res).float()
    a = (x.double() @ w.double().t()).to(BF).float()
    want = (res.float() + a).to(BF).float()
    bound = bf16_ulp(a) + 2 * bf16_ulp(torch.maximum(got.abs(), want.abs()))
    assert bool(((got - want).abs() <= bound).all())


# 33..64 rows: one row block of 64, 40 to 96 columns per workgroup and 1 to 8 K splits as the plan
# decides; without room for partials unsplit, in blocks of 16 to 40 columns
@pytest.mark.parametrize("name", list(SHAPES))
@pytest.mark.parametrize("M", [33, 47, 64])
def test_small_row_counts(ops, name, M):
    x, w, res = _operands(name, M)
    N, K = SHAPES[name]
    acc = x.double() @ w.double().t()
    a = acc.to(BF).float()
    for room in (True, False):
        ws = None if room else torch.zeros(256, dtype=torch.uint8, device="cuda")
        got = _linear(ops, name, x, w, res, ws=ws).float()
        if name == "gu":
            gate, up = a[:, :N], a[:, N:]
            sg = torch.sigmoid(gate)
            s = (gate * sg).to(BF).float()
            want = (s * up).to(BF).float()
            bound = (up.abs() * ((sg * (1 + gate * (1 - sg))).abs() * bf16_ulp(gate) + bf16_ulp(s))
                     + s.abs() * bf16_ulp(up) + 2 * bf16_ulp(torch.maximum(got.abs(), want.abs())) + 2 ** -12)
        elif name == "qkv":
            want = a
            bound = 2 * bf16_ulp(torch.maximum(got.abs(), want.abs())) + 2 ** -9
        else:
            want = (res.float() + a).to(BF).float()
            bound = bf16_ulp(a) + 2 * bf16_ulp(torch.maximum(got.abs(), want.abs()))
        assert bool(((got - want).abs() <= bound).all()), f"room {room}"


@pytest.mark.parametrize("name,M", [("gu", 47), ("o", 33), ("qkv", 300), ("gu", 601), ("down", 1500), ("o", 4095)])
def test_outputs_aligned_to_8_bytes(ops, name, M):
    """An output (and residual) whose rows start 8 bytes off a 16-byte boundary takes the narrow
    stores: the same bits, and nothing written beside the rows."""
    x, w, res = _operands(name, M)
    N = SHAPES[name][0]
    want = _linear(ops, name, x, w, res)
    buf = torch.full((M, N + 12), 7.0, dtype=BF, device="cuda")
    rbuf = torch.zeros((M, N + 12), dtype=BF, device="cuda")
    out, r2 = buf[:, 4:4 + N], rbuf[:, 4:4 + N]
    r2.copy_(res)
    _linear(ops, name, x, w, r2, out=out)
    assert torch.equal(out, want)
    assert bool((buf[:, :4] == 7).all()) and bool((buf[:, 4 + N:] == 7).all())


@pytest.mark.parametrize("kind,mt,nt", list(INSTANCES))
def test_every_instance(ops, kind, mt, nt):
    M, N, K = INSTANCES[kind, mt, nt]
    print(f"\n[case] {kind} {{{mt}, {nt}}}: {M} x {N} x {K}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    x = torch.empty((M, K), dtype=BF, device="cuda").normal_(0, 1, generator=g)
    for epi in (ops.EPI_SWIGLU,) if kind == "swiglu" else (ops.EPI_NONE, ops.EPI_RES):
        check_linear(ops, epi, x, N, g)


@pytest.mark.parametrize("B,S,N", [(33, 20, 4), (48, 40, 4), (100, 12, 3), (130, 9, 3)])
def test_decode_steps_with_split_partials(B, S, N):
    """Decode steps of more than 32 rows, whose projections leave K-split partials in the LM head's
    region: greedy ids under the margin rule against the oracle."""
    from engine import Engine
    from helpers import ORACLE_TIE, ensure_oracle_built, margin_rule
    from oracle import qwen3_ref as R
    from oracle import synth
    ensure_oracle_built()
    print(f"\n[case] decode B={B} S={S} N={N}", flush=True)
    eng = Engine.synthetic(n_layers=2, seed=1)
    eng.tree_mode = "0"
    prompt = synth.prompt_ids(60 + B, B, S)
    toks = torch.tensor(list(eng.generate(prompt.tolist(), N))).numpy().T
    tl = R.Qwen3Ref.from_synth(1, 2).teacher_logits(prompt, toks)
    assert margin_rule(toks, tl, margin=ORACLE_TIE, what=f"decode B={B}") == []


@pytest.mark.parametrize("B,S,N", [(40, 16, 3), (100, 9, 2)])
def test_decode_step_logits_with_split_partials(B, S, N):
    """The same steps by their logits (from the residual each step leaves), which see what greedy ids
    do not."""
    from engine import Engine
    from helpers import engine_step_logits, ensure_oracle_built
    from oracle import qwen3_ref as R
    from oracle import synth
    ensure_oracle_built()
    print(f"\n[case] decode logits B={B} S={S} N={N}", flush=True)
    eng = Engine.synthetic(n_layers=2, seed=1)
    eng.tree_mode = "0"
    prompt = synth.prompt_ids(80 + B, B, S)
    ids, arg, lg = engine_step_logits(eng, prompt, N)
    assert (ids == arg).all()
    want = R.Qwen3Ref.from_synth(1, 2).teacher_logits(prompt, ids).double()
    rel = (lg.double() - want).flatten(2).norm(dim=-1) / want.norm(dim=-1)
    print(f"relative error of the worst row and step {float(rel.max()):.4f}", flush=True)
    # bf16 roundings of 4 such layers move the logits by 1.9e-2 of their norm against 64 bits, those of
    # 2 by its square root's share; the engine and the oracle each
    assert float(rel.max()) <= 2 * 1.9e-2 * (2 / 4) ** 0.5
