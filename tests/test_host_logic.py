"""Host-side logic that runs without a GPU: synthetic checkpoints, config parsing, rope tables,
the cap rule, and the engine's refusal to run without a GPU."""
import tempfile

import pytest
import torch

from dryft_amd import synth
from dryft_amd.engine import CAP_GRAN, Engine, build_rope_tables, rope_theta
from oracle.reference import OracleEngine
from oracle.reference import build_rope_tables as oracle_rope


def test_synth_is_deterministic_and_named_like_hf():
    cfg = synth.qwen3_config(num_hidden_layers=2, vocab_size=512, hidden_size=256,
                             intermediate_size=192, num_attention_heads=8, num_key_value_heads=2)
    a = synth.random_weights(cfg, seed=3)
    b = synth.random_weights(cfg, seed=3)
    c = synth.random_weights(cfg, seed=4)
    assert a.keys() == b.keys()
    assert all(torch.equal(a[k], b[k]) for k in a)
    assert not torch.equal(a["model.embed_tokens.weight"], c["model.embed_tokens.weight"])
    assert a["model.layers.0.self_attn.q_proj.weight"].shape == (8 * 128, 256)
    assert a["model.layers.1.mlp.down_proj.weight"].shape == (256, 192)
    assert "lm_head.weight" not in a                      # tied
    w = a["model.layers.0.mlp.up_proj.weight"].float()
    assert abs(w.std().item() - 0.02) < 0.002 and abs(w.mean().item()) < 0.002
    n = a["model.layers.0.input_layernorm.weight"].float()
    assert abs(n.mean().item() - 1.0) < 0.01


def test_synth_roundtrip_through_safetensors():
    cfg = synth.qwen3_config(num_hidden_layers=1, vocab_size=256, hidden_size=128,
                             intermediate_size=64, num_attention_heads=2, num_key_value_heads=1)
    w = synth.random_weights(cfg, seed=0)
    d = tempfile.mkdtemp()
    synth.write_model(d, cfg, w)
    ref_dir = OracleEngine(d)
    ref_mem = OracleEngine.from_state_dict(cfg, w)
    assert torch.equal(ref_dir.layers[0].wqkv, ref_mem.layers[0].wqkv)
    # q | k | v order of the fused projection (engine.py:300-302)
    assert torch.equal(ref_mem.layers[0].wqkv[:256], w["model.layers.0.self_attn.q_proj.weight"])
    assert torch.equal(ref_mem.layers[0].wqkv[256:384], w["model.layers.0.self_attn.k_proj.weight"])
    assert torch.equal(ref_mem.lm_head, ref_mem.embed)


def test_rope_theta_both_config_forms():
    assert rope_theta({"rope_theta": 5e6}) == 5e6
    assert rope_theta({"rope_parameters": {"rope_theta": 1e6, "rope_type": "default"}}) == 1e6


def test_engine_rope_tables_are_the_oracle_bits():
    cos, sin = build_rope_tables(5e6, 128, 1024)
    rc, rs = oracle_rope(5e6, 128, 1024)
    assert torch.equal(cos, rc) and torch.equal(sin, rs)


def test_cap_rule():
    # engine.py:707: cap = ceil((S + n) / 128) * 128
    for S, n, cap in ((512, 32, 640), (2048, 1024, 3072), (1, 1, 128), (127, 1, 128), (128, 1, 256)):
        assert -(-(S + n) // CAP_GRAN) * CAP_GRAN == cap


def test_engine_refuses_cpu():
    with pytest.raises(RuntimeError):
        Engine.from_state_dict(synth.qwen3_config(num_hidden_layers=1), {}, device="cpu")


@pytest.mark.parametrize("nh,nkv", [(4, 1), (8, 2), (32, 8), (64, 8), (32, 16)])
def test_qkv_head_grouped_order(nh, nkv):
    """The fused step's raw q|k|v slot is head-grouped (per kv head: its nh / nkv q heads, then
    k, then v, 128 columns each). FusedStep.qkv_natural must map it back to cat(q, k, v): applied
    to the head-grouped order of the column indices it gives 0, 1, 2, ... and it keeps every head
    of a group next to its own k and v (head h of group g is q head g * nh / nkv + h)."""
    from dryft_amd.step import FusedStep
    hd = 128
    g = nh // nkv
    n = (nh + 2 * nkv) * hd
    # head-grouped order written out head by head (the layout the step's QKV phase writes)
    order = []
    for kv in range(nkv):
        for h in range(g):
            order += range((kv * g + h) * hd, (kv * g + h + 1) * hd)
        order += range((nh + kv) * hd, (nh + kv + 1) * hd)
        order += range((nh + nkv + kv) * hd, (nh + nkv + kv + 1) * hd)
    grouped = torch.tensor(order).view(1, 1, n)
    assert sorted(order) == list(range(n))
    assert torch.equal(FusedStep.qkv_natural(grouped, nh, nkv).view(-1), torch.arange(n))


def test_gemm_table_is_nowhere_much_slower_than_the_heuristic():
    """By its own timings the committed table's entries are at most 5% (and a timing's last digit) slower
    than the heuristic's first candidate, at three row counts of each entry's range and at the row counts
    between grid points that it records; the lookup takes the entry of the range."""
    import json
    from dryft_amd import hipops
    with open(hipops.GEMM_TABLE) as f:
        doc = json.load(f)
    table = hipops.load_gemm_table()
    for c in doc["check"].values():
        assert c["table_ms"] <= 1.06 * c["heuristic_first_ms"], c
    for key, rows in doc["shapes"].items():
        n, k = (int(v) for v in key.split("x"))
        assert [m for m, _ in rows] == doc["grid"]
        for (m, sol), prev in zip(rows, [16] + doc["grid"]):
            t = doc["timing_ms"][key][str(m)]
            assert all(a <= 1.05 * b + 2e-4 for a, b in zip(t["table"], t["heuristic_first"])), (key, m, t)
            assert {hipops.gemm_solution(table, n, k, v) for v in (prev + 1, m)} == {sol}
        assert hipops.gemm_solution(table, n, k, 10 ** 6) == rows[-1][1]


class FakeLib:
    """The library's side of HipOps on the CPU: sizes and choices as the library gives them, and the names
    of the kernels that would have been launched."""

    def __init__(self):
        self.launched = []

    def dd_linear_supported(self, M, N, K):
        return int(1 <= M <= 64 and N >= 1 and K >= 64 and K % 64 == 0)

    def __getattr__(self, name):
        if name.endswith(("_bytes", "_splitk", "_counters")):
            return lambda *a: 16
        return lambda *a: self.launched.append(name) or 0


@pytest.fixture
def cpu_ops(monkeypatch):
    """HipOps with its kernels replaced by a record of their launches, for CPU tensors."""
    from types import SimpleNamespace
    from dryft_amd import hipops
    ops = object.__new__(hipops.HipOps)
    ops.L, ops.e, ops.use_gemv, ops._gemm_table = FakeLib(), SimpleNamespace(eps=1e-6), True, {}
    monkeypatch.setattr(hipops, "_bf16_ok", lambda *ts: all(
        t.dtype == torch.bfloat16 and t.is_contiguous() for t in ts))
    monkeypatch.setattr(hipops, "_stream", lambda dev: 0)
    monkeypatch.setattr(ops, "_zeroed_counters", lambda n, dev: torch.zeros(n, dtype=torch.int32))
    monkeypatch.setattr(ops, "_gemm_workspace", lambda dev, stream: torch.empty(16, dtype=torch.uint8))
    return ops


@pytest.mark.parametrize("K", [192, 200])
@pytest.mark.parametrize("M", [1, 16, 17, 100])
def test_mismatched_operands_reach_no_kernel(cpu_ops, M, K):
    """Operands whose shapes do not fit raise, and nothing is launched that would read past them."""
    b = lambda *s: torch.ones(s, dtype=torch.bfloat16)  # noqa: E731
    x, w, h, n = b(M, K), b(80, K), b(M, 80), b(80)
    ops = cpu_ops
    products = [lambda: ops.linear(x, b(80, K - 64)), lambda: ops.linear(x, b(80, K + 8)),
                lambda: ops.gate_up_silu(x, b(80, K - 64)), lambda: ops.linear_add_norm(x, b(80, K - 64), h, n)]
    # here the product fits and may run; what follows it does not
    epilogues = [lambda: ops.gate_up_silu(x, b(81, K)), lambda: ops.linear_add_norm(x, w, b(M, 72), n),
                 lambda: ops.linear_add_norm(x, w, h, b(72)), lambda: ops.add_rms(h, b(M, 72), n),
                 lambda: ops.add_rms(h, h, b(72)), lambda: ops.rms(h, b(72)), lambda: ops.silu_mul(b(M, 81))]
    if M > 1:
        epilogues.append(lambda: ops.linear_add_norm(x, w, b(M + 1, 80), n))
    for calls, allowed in ((products, set()), (epilogues, {"dd_linear", "dd_gemv", "dd_gemm_bf16"})):
        for call in calls:
            ops.L.launched.clear()
            with pytest.raises(RuntimeError):
                call()
            assert set(ops.L.launched) <= allowed, ops.L.launched
    ops.L.launched.clear()
    for call in (ops.linear, ops.gate_up_silu, lambda x, w: ops.linear_add_norm(x, w, h, n)):
        call(x, w)
        assert ops.L.launched or M > 16                   # what fits still runs
        ops.L.launched.clear()


@pytest.mark.parametrize("M", [17, 64, 65, 255, 256, 300])
def test_products_are_seen_by_what_watches_torch(cpu_ops, monkeypatch, M):
    """Above 16 rows a product that gradients, function transforms, tracing, modes or tensor subclasses take
    part in stays F.linear; a plain one, also under torch.set_default_device, is the kernels'."""
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    g = torch.Generator().manual_seed(M)
    x, t = (torch.randint(-1, 2, (M, 64), generator=g).to(torch.bfloat16) for _ in range(2))
    w = torch.randint(-1, 2, (48, 64), generator=g).to(torch.bfloat16)
    linear, launched = cpu_ops.linear, cpu_ops.L.launched
    y, dy = x @ w.t(), t @ w.t()

    out, tangent = torch.func.jvp(lambda a: linear(a, w), (x,), (t,))
    assert torch.equal(out, y) and torch.equal(tangent, dy)
    with forward_ad.dual_level():
        out = forward_ad.unpack_dual(linear(forward_ad.make_dual(x, t), w))
        assert torch.equal(out.primal, y) and torch.equal(out.tangent, dy)
    assert torch.equal(torch.vmap(lambda a: linear(a, w))(torch.stack([x, t])), torch.stack([y, dy]))
    for mode in ("real", "fake"):
        assert torch.equal(make_fx(lambda a, b: linear(a, b), tracing_mode=mode)(x, w)(t, w), dy)
    assert torch.equal(torch.jit.trace(lambda a: linear(a, w), (x,), check_trace=False)(t), dy)
    torch._dynamo.reset()
    assert torch.equal(torch.compile(lambda a, b: linear(a, b), backend="eager", fullgraph=True)(x, w), y)
    with FlopCounterMode(display=False) as flops:
        linear(x, w)
    assert flops.get_total_flops() == 2 * M * 48 * 64

    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    with Mode():
        linear(x, w)
    assert torch.nn.functional.linear in seen
    assert type(linear(x.as_subclass(Sub), w)) is Sub
    weight = torch.nn.Parameter(w)
    linear(x, weight).backward(t[:, :48])
    assert weight.grad is not None and not launched
    if M < 256:
        with monkeypatch.context() as m:
            m.setattr(torch, "is_autocast_enabled", lambda device: True)
            m.setattr(torch, "get_autocast_dtype", lambda device: torch.float16)
            linear(x, w)
        assert not launched
    torch.set_default_device("cpu")
    try:
        linear(x, w)
    finally:
        torch.set_default_device(None)
    with torch.no_grad():
        linear(x, weight)
    assert launched == ["dd_linear" if M <= 64 else "dd_gemm_bf16"] * 2


def test_op_counters_are_not_shared(monkeypatch):
    """Calls on two streams, and calls of two graph captures, never get the same counters (calls that
    overlap would race on them); one stream, and one capture on one stream, keeps its own."""
    from dryft_amd import hipops
    at = {"stream": 1, "capture": 0}

    class Lib:
        @staticmethod
        def dd_capture_id(stream, out):
            out._obj.value = at["capture"]
            return 0

    ops = object.__new__(hipops.HipOps)
    ops.L, ops._counters, ops._graph_counters = Lib, {}, (0, {})
    ops.err = torch.zeros(1)
    ops._spares = torch.zeros(3, hipops.COUNTERS, dtype=torch.int32)
    ops._spare = list(ops._spares)
    monkeypatch.setattr(hipops, "_stream", lambda dev: at["stream"])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: at["capture"] != 0)

    def get(stream, capture, n=8):
        at.update(stream=stream, capture=capture)
        c = ops._zeroed_counters(n, torch.device("cpu"))
        assert c.numel() >= n and not c.any()
        return c

    a, b = get(1, 0), get(2, 0)
    g1, g1_side, = get(3, 7), get(4, 7)
    assert get(3, 7) is g1                          # before another capture begins
    g2 = get(3, 8)
    assert get(1, 0) is a and get(2, 0) is b and get(3, 8) is g2
    kept = [a, b, g1, g1_side, g2, get(3, 0), get(1, 0, 20000), get(3, 9), get(3, 9, 20000), get(3, 10)]
    assert len({c.data_ptr() for c in kept}) == len(kept)
    for s in range(300):                            # bounded
        get(100 + s, 0)
    assert len(ops._counters) <= hipops.COUNTERS_MAX
