"""The Sebesun design in the engine against the plain implementation (tests/plain_sebesun.py).

Without a GPU: the configuration, its description as parts and the loader's binding.  On the GPU: every mechanism
alone (one-layer models and the kernels called directly with inputs made so that one far token decides the result),
whole prompts, prompts cut into portions down to two tokens, prefill against token-by-token decoding, batches of
unequal requests against each alone, slots and pages that are used again, long decoding over several pages, the
first tokens of a sequence, and greedy generation through ``generate``.  In float32 and in bfloat16.
"""
import math

import numpy as np
import pytest
import torch

import plain_sebesun as P
import sebesun_tiny as S
import tiny
from palm_infra_amd.config import ConfigError, config_from_dict

gpu = pytest.mark.gpu
DTYPES = ("float32", "bfloat16")
LENGTHS = {"P": [1, 2, 63, 64, 65, 130, 200, 17], "Q": [129, 3, 70, 64, 1, 191], "R": [5, 66, 128, 31]}


# ---- without a GPU ---------------------------------------------------------------------------------------

def test_registry_picks_the_design_by_its_config_key():
    cfg = config_from_dict(S.CONFIGS["P"])
    assert type(cfg).__name__ == "SebesunConfig" and cfg.architecture == "Sebesun"
    assert config_from_dict(cfg.to_dict()) == cfg


def test_spec_names_every_tensor_with_its_shape():
    spec = config_from_dict(S.CONFIGS["Q"]).spec()
    exp = spec.expected_tensors()
    assert exp["embed"][0] == (130, 48) and exp["head"][0] == (130, 48) and exp["final.norm"][0] == (48,)
    assert exp["l0.mix.x"][0] == (1 + 2 * 17, 40) and exp["l0.mix.conv"][0] == (40, 2) and exp["l0.mix.A_log"][0] == (40, 17)
    assert exp["l1.mix.q"][0] == (3 * 2 * 24, 48) and exp["l1.mix.k"][0] == (3 * 2 * 24, 48) and exp["l1.mix.v"][0] == (3 * 20, 48)
    assert exp["l3.mix.k"][0] == (1 * 2 * 8, 48) and exp["l3.mix.o"][0] == (48, 2 * 72) and exp["l3.mlp.act"][0] == (2,)
    assert exp["l2.mix.g"][0] == (80, 48) and "l2.norm2" not in exp and "l3.norm2" in exp
    assert [exp[f"l{i}.dwa"][0] for i in range(5)] == [(2,), (3,), (4,), (5,), (6,)]
    assert spec.keeps_results


def test_cache_needs_follow_the_layers():
    from palm_infra_amd.cache import KVNeed, StateNeed
    from palm_infra_amd.parts import cache_needs
    spec = config_from_dict(S.CONFIGS["Q"]).spec()
    needs = [cache_needs(layer) for layer in spec.layers]
    assert needs[0] == [StateNeed("scan", (40, 17)), StateNeed("conv", (1, 40))]
    assert needs[1] == [KVNeed(6, 24, None, value_heads=3, value_dim=20)]
    assert needs[2] == [StateNeed("retention", (1, 24, 80))]
    assert needs[4] == [StateNeed("scan", (72, 33)), StateNeed("conv", (0, 72))]


@pytest.mark.parametrize("change,what", [
    (lambda c: c["layers"][0].update(type="lstm"), "type"),
    (lambda c: c["layers"][0]["mixer"].update(kv_heads=3), "multiple"),
    (lambda c: c["layers"][1]["mixer"].update(decay=[0.5]), "decay"),
    (lambda c: c["layers"][1]["mixer"].update(rot={"dims": 7, "base": 10.0}), "rot"),
    (lambda c: c["layers"][2]["mlp"].update(kind="routed"), "dense"),
    (lambda c: c.pop("width"), "width"),
    (lambda c: c["norm"].pop("eps"), "eps"),
])
def test_bad_configurations_are_refused(change, what):
    import copy
    raw = copy.deepcopy(S.CONFIGS["P"])
    change(raw)
    with pytest.raises(ConfigError, match=what):
        config_from_dict(raw)


def test_random_model_folder_is_read_by_the_plain_implementation(tmp_path):
    from palm_infra_amd.weights import write_random_model
    d = write_random_model(S.CONFIGS["R"], 5, tmp_path / "m", "bfloat16")
    cfg, w = P.read_model(d)
    assert cfg["layers"][0]["type"] == "retention" and w["l0.mix.q"].shape == (64, 40) and w["l0.mix.v"].shape == (96, 40)
    logits = P.forward(cfg, w, [1, 2, 3])
    assert logits.shape == (3, 97) and torch.isfinite(logits).all()


def test_plain_retention_equals_its_sum_over_the_past():
    """The oracle's recurrence against the closed form o_t = sum_(s<=t) decay^(t-s) (q_t . k_s) v_s."""
    torch.manual_seed(0)
    m = {"heads": 2, "dim": 6, "vdim": 5, "decay": [0.9, 0.7], "rot": {"dims": 4, "base": 50.0}}
    W, T = 10, 9
    w = {"q": torch.randn(12, W, dtype=P.F64), "k": torch.randn(12, W, dtype=P.F64), "v": torch.randn(10, W, dtype=P.F64),
         "g": torch.randn(10, W, dtype=P.F64), "o": torch.eye(10, dtype=P.F64)}
    h = torch.randn(T, W, dtype=P.F64)
    got = P.retention(h, w, "", m, 1e-6)
    q = P.rotate_half_split((h @ w["q"].T).view(T, 2, 6), 4, 50.0)
    k = P.rotate_half_split((h @ w["k"].T).view(T, 2, 6), 4, 50.0) * 6 ** -0.5
    v = (h @ w["v"].T).view(T, 2, 5)
    o = torch.zeros(T, 2, 5, dtype=P.F64)
    for hd in range(2):
        for t in range(T):
            for s in range(t + 1):
                o[t, hd] += m["decay"][hd] ** (t - s) * (q[t, hd] @ k[s, hd]) * v[s, hd]
    want = P.unit_rms(o, 1e-6).reshape(T, 10) * P.silu(h @ w["g"].T)
    assert torch.allclose(got, want, atol=1e-10)


# ---- engines and references ------------------------------------------------------------------------------

_dirs, _engines, _refs = {}, {}, {}


def model_dir(tmp_path_factory, name: str, store: str):
    key = (name, store)
    if key not in _dirs:
        raw = S.CONFIGS.get(name) or S.SINGLE[name]
        _dirs[key] = S.write_model(raw, S.SEEDS.get(name, 21), tmp_path_factory.mktemp(f"sebesun_{name}_{store}"), store)
    return _dirs[key]


def engine_for(tmp_path_factory, name: str, dtype: str, **options):
    from palm_infra_amd.engine import Engine
    key = (name, dtype, tuple(sorted(options.items())))
    if key not in _engines:
        _engines[key] = Engine.from_dir(model_dir(tmp_path_factory, name, dtype), dtype=dtype, max_tokens=64 * 24, **options)
    return _engines[key]


def reference(tmp_path_factory, name: str, dtype: str, ids):
    key = (name, dtype, tuple(ids))
    if key not in _refs:
        cfg, w = P.read_model(model_dir(tmp_path_factory, name, dtype))
        _refs[key] = P.forward(cfg, w, ids)
    return _refs[key]


def assert_close(got, ref, dtype: str, what: str = "") -> None:
    """float32: 1e-4 absolute on logits of order one, the gate that shows faults.  bfloat16: a row's root mean square
    error within a fifth of the logits' scale, all rows together within a twentieth, an element within three quarters.
    A row here or there may break these by rounding alone: the q and k norms divide by the root mean square of a
    projection of as few as 8 values, which now and then is small against the rounding of its input (one row in some
    thousand was off by half the scale with float32 twins exact everywhere).  So one row in a hundred (at least one) may
    be over the row gate, but never by more than the scale itself, and the other gates hold for the rest."""
    if dtype == "float32":
        return tiny.assert_logits_close(got, ref, dtype, what)
    got = torch.as_tensor(got).double().cpu().reshape(ref.shape)
    assert torch.isfinite(got).all(), f"{what}: logits are not finite"
    err = (got - ref.double()).abs().reshape(-1, ref.shape[-1])
    scale = float(ref.double().pow(2).mean().sqrt())
    rows = err.pow(2).mean(-1).sqrt()
    over = rows > 0.2 * scale
    assert int(over.sum()) <= max(1, rows.numel() // 100), (f"{what}: bfloat16 rms error over a fifth of {scale:.3e} in "
                                                             f"{int(over.sum())} of {rows.numel()} rows, the worst {float(rows.max()):.3e} in row {int(rows.argmax())}")
    assert float(rows.max()) <= scale, f"{what}: bfloat16 rms error {float(rows.max()):.3e} in row {int(rows.argmax())} vs {scale:.3e}"
    rest = err[~over]
    if rest.shape[0] >= 16:
        assert float(rest.pow(2).mean().sqrt()) <= 0.05 * scale, f"{what}: bfloat16 rms error over all rows vs {scale:.3e}"
    if rest.numel():
        assert float(rest.max()) <= 0.75 * scale, f"{what}: bfloat16 max error {float(rest.max()):.3e} vs {scale:.3e}"


class Pool:
    """Rows checked a few at a time, then all together (the gate over all rows needs many)."""

    def __init__(self, dtype, what):
        self.dtype, self.what, self.got, self.ref = dtype, what, [], []

    def add(self, got, ref):
        got = torch.as_tensor(got).double().cpu().reshape(ref.shape)
        assert_close(got, ref, self.dtype, self.what)
        self.got.append(got.reshape(-1, ref.shape[-1]))
        self.ref.append(ref.double().reshape(-1, ref.shape[-1]))

    def check(self):
        assert_close(torch.cat(self.got), torch.cat(self.ref), self.dtype, self.what + " (all rows together)")


def raw_of(name):
    return S.CONFIGS.get(name) or S.SINGLE[name]


CASES = [(n, d) for n in ("P", "Q", "R") for d in DTYPES]


# ---- every mechanism alone -------------------------------------------------------------------------------

@gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", sorted(S.SINGLE))
def test_one_layer_of_one_kind(tmp_path_factory, kind, dtype):
    from palm_infra_amd.engine import StepEntry
    eng = engine_for(tmp_path_factory, kind, dtype)
    for ids in S.prompts(raw_of(kind), [1, 9, 64, 131]):
        slot = eng.open()
        got = eng.step([StepEntry(slot, ids, list(range(len(ids))))])
        eng.close(slot)
        assert_close(got, reference(tmp_path_factory, kind, dtype, ids), dtype, f"{kind} alone, {len(ids)} tokens")


@gpu
@pytest.mark.parametrize("W", [50, 64, 2048, 5000, 20000])      # no multiple of four, narrow, wide, several groups a thread, beyond them
def test_stream_kernel_norms_adds_and_averages_over_depth(W):
    from palm_infra_amd.kernels import ops
    torch.manual_seed(1)
    n, J = 7, 3
    x = torch.randn(n, W, device="cuda")
    y = torch.randn(n, W, device="cuda") * 3
    w = torch.rand(W, device="cuda") + 0.5
    results = torch.randn(J + 2, n, W, device="cuda")
    mix = torch.randn(J + 1, device="cuda")
    for delta in (y, y.bfloat16()):
        d64 = delta.double()
        summed = x.double() + P.rms_norm(d64, w.double(), 1e-5)
        want = sum(mix[j].double() * results[j].double() for j in range(J)) + mix[J].double() * summed
        xs, rs = x.clone(), results.clone()
        h = ops.add_normed(xs, delta, w, 1e-5, torch.bfloat16, results=rs, mix=mix)
        assert torch.allclose(xs.double(), want, atol=1e-5) and torch.allclose(rs[J].double(), summed, atol=1e-5)
        assert torch.equal(rs[J + 1], results[J + 1]) and torch.equal(rs[:J], results[:J])
        assert torch.equal(h, xs.bfloat16())
        xs = x.clone()
        assert ops.add_normed(xs, delta, w, 1e-5, torch.float32) is xs
        assert torch.allclose(xs.double(), summed, atol=1e-5)


@gpu
@pytest.mark.parametrize("W,J", [(4096, 0), (4096, 4), (4100, 5), (8192, 8), (12288, 7), (16384, 1)])
def test_averages_over_many_planes(W, J):
    """One to four groups of four a thread, and planes that fill the reads under way together or leave some over."""
    from palm_infra_amd.kernels import ops
    torch.manual_seed(W + J)
    n = 3
    x, y, w = torch.randn(n, W, device="cuda"), torch.randn(n, W, device="cuda") * 3, torch.rand(W, device="cuda") + 0.5
    results, mix = torch.randn(J + 2, n, W, device="cuda"), torch.randn(J + 1, device="cuda")
    summed = x.double() + P.rms_norm(y.double(), w.double(), 1e-5)
    want = sum((mix[j].double() * results[j].double() for j in range(J)), mix[J].double() * summed)
    xs, rs = x.clone(), results.clone()
    h = ops.add_normed(xs, y, w, 1e-5, torch.bfloat16, results=rs, mix=mix)
    assert torch.allclose(xs.double(), want, atol=1e-5) and torch.allclose(rs[J].double(), summed, atol=1e-5)
    assert torch.equal(rs[J + 1], results[J + 1]) and torch.equal(rs[:J], results[:J]) and torch.equal(h, xs.bfloat16())


@gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("lens,C,wide", [([16], 64, 64), ([1, 15, 47], 1028, 2060), ([33, 2, 130], 260, 264), ([40, 3], 66, 66), ([20, 16], 64, 67),
                                         ([1, 15, 47, 16, 33], 11800, 11804), ([16, 130], 9204, 18408), ([47] + [1] * 20, 8500, 8504), ([60, 50], 12000, 12001)])
def test_causal_conv_in_runs_is_the_convolution_token_by_token(dtype, taps, lens, C, wide):
    """Runs of tokens a thread, their remainders, and the sizes that go a token a thread: bit for bit the steps of one token each."""
    from palm_infra_amd.kernels import ops
    from palm_infra_amd.parts import make_context
    torch.manual_seed(taps * C + wide)
    x = torch.randn(sum(lens), wide, device="cuda").to(dtype)
    w, bias = torch.randn(C, taps, device="cuda"), torch.randn(C, device="cuda") if C % 64 == 0 else None
    before = torch.randn(len(lens), taps - 1, C, device="cuda")
    slots = list(range(len(lens)))[::-1]
    state = before.clone()
    got = ops.causal_conv(x, C, w, bias, state, make_context(slots, [0] * len(lens), [[0] * n for n in lens], dtype, "cuda"))
    ends = [sum(lens[:b + 1]) for b in range(len(lens))]
    for b, n in enumerate(lens):
        one = before.clone()
        ctx = make_context([slots[b]], [0], [[0]], dtype, "cuda")
        for t in range(n):
            row = ends[b] - n + t
            assert torch.equal(ops.causal_conv(x[row:row + 1], C, w, bias, one, ctx)[0], got[row]), (b, t)
        assert torch.equal(one[slots[b]], state[slots[b]])


@gpu
def test_xielu_on_both_sides_of_zero():
    from palm_infra_amd.kernels import ops
    z = torch.linspace(-12, 12, 1001, device="cuda")
    for p, q in ((0.3, -0.7), (-2.0, 1.5), (25.0, 0.0)):
        pq = torch.tensor([p, q], device="cuda")
        want = P.xielu(z.double().cpu(), torch.tensor(p, dtype=P.F64), torch.tensor(q, dtype=P.F64))
        got = ops.xielu(z, pq).double().cpu()
        assert torch.allclose(got, want, rtol=2e-6, atol=2e-6)
    assert float(ops.xielu(torch.zeros(1, device="cuda"), torch.tensor([0.3, 0.2], device="cuda"))) == 0.0


@gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 7, 8, 4095, 4100, 70001])
def test_xielu_in_pieces_of_sixteen_bytes(dtype, n):
    """Every remainder and operands that do not start on 16 bytes, around zero, at a half and far out: 32-bit arithmetic of some
    roundings, and one to the type."""
    from palm_infra_amd.kernels import ops
    g = torch.Generator().manual_seed(n)
    z = torch.randn(n + 1, generator=g) * torch.tensor([1e-4, 0.5, 1.0, 30.0, 3000.0])[torch.randint(0, 5, (n + 1,), generator=g)]
    z[:4] = torch.tensor([-0.5, -0.49999, -0.50001, 0.0])[:n + 1]
    z, pq = z.to(dtype).cuda(), torch.tensor([0.3, -0.7], device="cuda")
    for part in (z[:n], z[1:]):
        want = P.xielu(part.double().cpu(), torch.tensor(0.3, dtype=P.F64), torch.tensor(-0.7, dtype=P.F64))
        got = ops.xielu(part, pq)
        # the two terms below zero cancel where they meet: some roundings of 2^-24 of the larger, |z| at most, and of the result
        bound = 16 * 2.0 ** -24 * (want.abs() + part.double().cpu().abs()) + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0)
        assert bool(((got.double().cpu() - want).abs() <= bound).all()), float(((got.double().cpu() - want).abs() / bound).max())
    odd = torch.tensor([float("nan"), float("inf"), float("-inf"), -3e38, -0.0], device="cuda")
    got = ops.xielu(odd, pq).cpu()
    assert torch.isnan(got[0]) and got[1] == float("inf") and torch.isnan(got[2]) and bool(torch.isfinite(got[3])) and got[4] == 0.0


@gpu
def test_xielu_below_zero_is_as_exact_as_its_exponential():
    """A steep negative side shows exp(z) - 1 - z itself: off by the exponential's last place, the difference's and the result's rounding."""
    from palm_infra_amd.kernels import ops
    g = torch.Generator().manual_seed(0)
    z = -torch.cat([torch.rand(1 << 18, generator=g) * top for top in (0.5, 1.0, 2.0, 20.0)])
    steep = 100.5                                             # 0.5 + softplus(100)
    got = ops.xielu(z.cuda(), torch.tensor([0.0, 100.0], device="cuda")).double().cpu().numpy()
    d = z.double().numpy()
    near = np.expm1(d)
    want = steep * (near - d) + 0.5 * d
    ulp = lambda x: np.spacing(np.abs(x).astype(np.float32)).astype(np.float64)
    bound = steep * (ulp(near) + 0.5 * ulp(near - d)) + 0.5 * ulp(want)
    assert (np.abs(got - want) <= bound).all(), float((np.abs(got - want) / bound).max())


def _step_context(lengths_before, new_counts, n_slots=None):
    """A cache-less context for kernels that only need the packed layout: slots 0.., given starts."""
    from palm_infra_amd.parts import make_context
    slots = list(range(len(new_counts)))
    return make_context(slots, list(lengths_before), [[0] * c for c in new_counts], torch.float32, "cuda")


@gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_retention_kernel_keeps_a_far_token_and_forgets_at_its_decay(dtype):
    """One early token has a large key that the last query is aligned with: among some hundred tokens it decides the
    output, scaled by decay^(distance).  The same rows in one step, and cut into portions of 2, 5 and 64 tokens."""
    from palm_infra_amd.kernels import ops
    torch.manual_seed(2)
    H, dk, dv, T, far = 2, 12, 20, 300, 3
    rows = (torch.randn(T, H * (2 * dk + 2 * dv)) * 0.3)
    direction = torch.randn(dk)
    rows[far, H * dk:H * dk + dk] = direction * 150.0            # k of head 0 at the far token
    rows[T - 1, 0:dk] = direction * 5.0                          # q of head 0 at the last token
    rows = rows.to(dtype).cuda()
    decay = torch.tensor([0.99, 0.9], device="cuda")
    r64 = rows.double().cpu()
    q, k = r64[:, :H * dk].view(T, H, dk), r64[:, H * dk:2 * H * dk].view(T, H, dk) * dk ** -0.5
    v, g = r64[:, 2 * H * dk:2 * H * dk + H * dv].view(T, H, dv), r64[:, 2 * H * dk + H * dv:]
    o = torch.zeros(T, H, dv, dtype=P.F64)
    for hd in range(H):
        Sm = torch.zeros(dk, dv, dtype=P.F64)
        for t in range(T):
            Sm = float(decay[hd]) * Sm + torch.outer(k[t, hd], v[t, hd])
            o[t, hd] = Sm.T @ q[t, hd]
    want = P.unit_rms(o, 1e-6).reshape(T, H * dv) * P.silu(g)
    # the far token carries the last row of head 0: without it the direction of o changes
    without = o[T - 1, 0] - 0.99 ** (T - 1 - far) * (q[T - 1, 0] @ k[far, 0]) * v[far, 0]
    assert without.norm() < 0.3 * o[T - 1, 0].norm()
    tol = 2e-5 if dtype == torch.float32 else 3e-2
    final = None
    # (tokens a step, tokens a chunk inside the kernel: None = its own choice, 0 = no chunks)
    for portion, chunk in ((T, 0), (T, None), (T, 32), (T, 104), (150, 64), (64, 0), (5, None), (2, None)):
        state = torch.zeros(2, H, dk, dv, device="cuda")
        got = []
        for lo in range(0, T, portion):
            n = min(portion, T - lo)
            ctx = _step_context([lo], [n])
            got.append(ops.retention(rows[lo:lo + n].contiguous(), H, dk, dv, decay, dk ** -0.5, 1e-6, state, ctx, chunk=chunk))
        got = torch.cat(got).double().cpu()
        assert (got - want).abs().max() < tol, f"portion {portion}, chunk {chunk}: {(got - want).abs().max()}"
        assert torch.count_nonzero(state[1]) == 0                 # the other slot's state is not touched
        final = state[0].clone() if final is None else final
        assert torch.allclose(state[0], final, rtol=1e-4, atol=1e-4), f"portion {portion}, chunk {chunk}: the state left behind differs"
    assert ops.retention_chunk(1, 2, 300) > 0 and ops.retention_chunk(1, 2, 300) < 300      # the second case above did cut


@gpu
@pytest.mark.parametrize("dk,dv", [(64, 128), (64, 256), (128, 128), (128, 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_retention_in_chunks_on_the_matrix_cores(dtype, dk, dv):
    """Runs of tokens around the borders of tiles and chunks, side by side in one step on states that hold something, against
    the recurrence in 64 bits and against the walk token by token: outputs with the per-head norm, outputs joined, the states."""
    from palm_infra_amd.kernels import ops
    torch.manual_seed(dk + dv)
    H, lengths = 3, [1, 16, 17, 64, 65, 130, 8]
    T, width = sum(lengths), 2 * dk + 2 * dv
    rows = (torch.randn(T, H * width + 8) * 0.5).to(dtype)
    decay = torch.tensor([0.97, 0.9, 0.999])
    state0 = torch.randn(len(lengths), H, dk, dv)
    weight = torch.rand(H * dv) + 0.5
    r64 = rows.double()[:, 8:]
    q, k = r64[:, :H * dk].view(T, H, dk), r64[:, H * dk:2 * H * dk].view(T, H, dk) * dk ** -0.5
    v, g = r64[:, 2 * H * dk:2 * H * dk + H * dv].view(T, H, dv), r64[:, 2 * H * dk + H * dv:]
    o, left, at = torch.zeros(T, H, dv, dtype=P.F64), [], 0
    for b, n in enumerate(lengths):
        S = state0[b].double()
        for t in range(at, at + n):
            S = decay.double()[:, None, None] * S + k[t][:, :, None] * v[t][:, None, :]
            o[t] = (S * q[t][:, :, None]).sum(1)
        left.append(S)
        at += n
    flat = o.reshape(T, H * dv)
    want = {"head": P.unit_rms(o, 1e-6).reshape(T, H * dv) * P.silu(g), "joined": P.unit_rms(flat, 1e-6) * weight.double() * torch.sigmoid(g)}
    # outputs of unit scale: 32-bit sums of up to 130 * dk terms, then one rounding to the type
    tol = 1e-4 if dtype == torch.float32 else 3e-2
    assert ops.recurrent().palm_retention_matrix_pays(H, dk, dv, len(lengths), T, max(lengths))
    for kind in ("head", "joined"):
        results = []
        for chunk in (None, 0):
            state = state0.clone().cuda()
            ctx = _step_context([0] * len(lengths), lengths)
            got = ops.retention(rows.cuda(), H, dk, dv, decay.cuda(), dk ** -0.5, 1e-6, state, ctx, chunk=chunk, col0=8,
                                joined_norm=weight.cuda() if kind == "joined" else None, gate_sigmoid=kind == "joined")
            error = (got.double().cpu() - want[kind]).abs().max()
            assert error < tol * max(1.0, float(want[kind].abs().max())), f"{kind}, chunk {chunk}: {error}"
            assert (state.double().cpu() - torch.stack(left)).abs().max() < 1e-4, f"{kind}, chunk {chunk}: the state"
            results.append(got)
        assert (results[0].float() - results[1].float()).abs().max() < tol * max(1.0, float(want[kind].abs().max()))


def test_which_steps_of_retention_go_in_chunks():
    """Not where many states would move for a few short runs: there the walk, which touches a state once, is the faster one."""
    from palm_infra_amd.kernels import ops
    pays = lambda lengths, heads=16, dim=128, vdim=256: bool(ops.recurrent().palm_retention_matrix_pays(heads, dim, vdim, len(lengths), sum(lengths), max(lengths)))
    assert pays([16]) and not pays([15]) and pays([2048]) and pays([1] * 8 + [300]) and pays([300] * 8) and pays([1] * 63 + [512])
    assert not pays([1] * 63 + [16]) and not pays([1] * 63 + [64]) and not pays([17] * 64) and not pays([24] * 128)
    assert pays([16] * 8, 32, 64, 128) and not pays([1] * 127 + [40], 32, 64, 128) and pays([24] * 32, 20, 128, 128)
    assert pays([700, 1], 1, 64, 256) and not pays([700, 1], 1, 64, 192) and not pays([700, 1], 1, 72, 128)


@gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lengths", [[1] * 40 + [20], [1] * 40 + [90]])
def test_retention_of_many_single_tokens_beside_a_run(dtype, lengths):
    """A run short enough that the step is walked over and one long enough that it goes in chunks: both against the walk."""
    from palm_infra_amd.kernels import ops
    torch.manual_seed(len(lengths))
    H, dk, dv, n, T = 16, 128, 256, len(lengths), sum(lengths)
    assert bool(ops.recurrent().palm_retention_matrix_pays(H, dk, dv, n, T, max(lengths))) == (lengths[-1] > 64)
    rows, decay, state0 = (torch.randn(T, H * (2 * dk + 2 * dv)) * 0.5).to(dtype).cuda(), torch.linspace(0.9, 0.999, H).cuda(), torch.randn(n, H, dk, dv).cuda()
    got, walked = [], []
    for results, chunk in ((got, None), (walked, 0)):
        state = state0.clone()
        results += [ops.retention(rows, H, dk, dv, decay, dk ** -0.5, 1e-6, state, _step_context([0] * n, lengths), chunk=chunk).float(), state]
    # 32-bit sums in another order, then one rounding to the type
    assert (got[0] - walked[0]).abs().max() < (1e-4 if dtype == torch.float32 else 2.0 ** -7) * float(walked[0].abs().max())
    assert (got[1] - walked[1]).abs().max() < 1e-4
    assert lengths[-1] > 64 or (torch.equal(got[0], walked[0]) and torch.equal(got[1], walked[1]))


def test_retention_starts_have_bounded_room():
    from palm_infra_amd.kernels import ops
    places = ops.recurrent().palm_retention_places
    assert places(16, 128, 256, 32768, 1) * 16 * 128 * 256 * 4 <= 128 << 20
    assert places(16, 128, 256, 700, 3) == 700 // 64 + 3 and places(1, 64, 128, 5, 1) == 1
    assert places(4096, 128, 256, 300, 2) == 1


@gpu
@pytest.mark.parametrize("lengths", [[700, 1, 500, 130], [1500], [20] * 70 + [1, 900]])
def test_retention_in_windows_of_chunks(lengths):
    """More chunks than the starts have room for: the state crosses from one window to the next, within a sequence and between
    sequences; against the walk token by token."""
    from palm_infra_amd.kernels import ops
    torch.manual_seed(len(lengths))
    H, dk, dv, T = 64, 128, 256, sum(lengths)
    assert ops.recurrent().palm_retention_places(H, dk, dv, T, len(lengths)) == 16 < T // 64 + len(lengths)
    assert ops.recurrent().palm_retention_matrix_pays(H, dk, dv, len(lengths), T, max(lengths))
    rows = (torch.randn(T, H * (2 * dk + 2 * dv)) * 0.5).bfloat16().cuda()
    decay, state0 = torch.linspace(0.9, 0.999, H).cuda(), torch.randn(len(lengths), H, dk, dv).cuda()
    results = []
    for chunk in (None, 0):
        state = state0.clone()
        y = ops.retention(rows, H, dk, dv, decay, dk ** -0.5, 1e-6, state, _step_context([0] * len(lengths), lengths), chunk=chunk)
        results.append((y.float(), state))
    (got, left), (want, walked) = results
    # one rounding to bfloat16 each; 32-bit sums in another order
    assert (got - want).abs().max() < 2.0 ** -7 * float(want.abs().max()) and (left - walked).abs().max() < 1e-4


@gpu
@pytest.mark.parametrize("dk,dv", [(64, 128), (128, 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("input_silu", [False, True])
def test_retention_chunks_keep_infinities_where_they_are(dtype, dk, dv, input_silu):
    """An infinite or no number in a token's values or keys reaches that token and later ones of its sequence, in its own value
    dimensions (or rows of the state) and no others, as when the tokens are walked over one by one; with the inputs through silu too."""
    from palm_infra_amd.kernels import ops
    torch.manual_seed(dk)
    H, lengths = 2, [40, 17, 70, 33]
    T = sum(lengths)
    rows = (torch.randn(T, H * (2 * dk + 2 * dv)) * 0.5).to(dtype)
    v0, inf = 2 * H * dk, float("inf")
    rows[21, v0 + 5] = inf                                   # sequence 0, token 21 (the middle of a block of sixteen), head 0
    rows[56, v0 + dv + 9] = float("nan")                     # sequence 1, its last token (the chunk ends there), head 1
    rows[57 + 66, v0 + 3] = inf                              # sequence 2, the second chunk
    rows[T - 1, H * dk + 7] = inf                            # sequence 3: a key of its last token, head 0
    decay, state0 = torch.tensor([0.97, 0.9]), torch.randn(len(lengths), H, dk, dv)
    results = []
    for chunk in (None, 0):
        state = state0.clone().cuda()
        ctx = _step_context([0] * len(lengths), lengths)
        raw = ops.retention(rows.cuda(), H, dk, dv, decay.cuda(), dk ** -0.5, 1e-6, state, ctx, chunk=chunk, input_silu=input_silu)
        results.append((raw.float().cpu(), state.cpu()))
    (got, left), (want, walked) = results
    # (the norm over a head's outputs spreads one of them over its head: a token's head is finite or it is not)
    whole = lambda y: torch.isfinite(y.view(T, H, dv)).all(-1)
    assert torch.equal(whole(got), whole(want)) and not whole(want).all()
    assert whole(got)[:21].all() and whole(got)[40:56].all() and whole(got)[57:57 + 66].all() and whole(got)[-33:-1].all()
    tol = 1e-4 if dtype == torch.float32 else 3e-2
    keep = whole(want)
    a, b = got.view(T, H, dv)[keep], want.view(T, H, dv)[keep]
    assert (a - b).abs().max() < tol * max(1.0, float(b.abs().max()))
    assert torch.equal(torch.isfinite(left), torch.isfinite(walked)) and not torch.isfinite(walked).all()
    assert (left[torch.isfinite(left)] - walked[torch.isfinite(walked)]).abs().max() < 1e-4


@gpu
@pytest.mark.parametrize("C,N", [(130, 3), (65, 8), (200, 16), (70, 20), (37, 64), (9, 100), (6, 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_selective_scan_alone(dtype, C, N):
    """Every build of the kernel by state size, around the borders of its tiles of sixteen tokens, on states that hold something, against
    the recurrence in 64 bits; a decay so fast that nothing stays, and an A that is no number, which its channel shows."""
    from palm_infra_amd.kernels import ops
    g = torch.Generator().manual_seed(C + N)
    lengths = [1, 15, 16, 17, 49, 2]
    T = sum(lengths)
    R = lambda *s: torch.randn(*s, generator=g)
    u, xz, bc = (R(T, c).to(dtype) for c in (C, 2 * C, 2 * N + 3))
    dtl, bias, skip, state0 = R(T, C), R(C) - 2.0, R(C), R(len(lengths), C, N)
    a_log = torch.log(torch.arange(1, N + 1).float()).repeat(C, 1) + 0.1 * R(C, N)
    a_log[1, 1], a_log[2, 2], a_log[4, 0] = 75.0, 88.7, float("nan")
    A, dt = -torch.exp(a_log.double()), torch.nn.functional.softplus((dtl + bias).double())
    z, B, Cm = xz[:, C:].double(), bc[:, 1:1 + N].double(), bc[:, 2 + N:2 + 2 * N].double()
    want, left, at = torch.zeros(T, C, dtype=P.F64), [], 0
    for b, n in enumerate(lengths):
        S = state0[b].double()
        for t in range(at, at + n):
            S = torch.exp(dt[t][:, None] * A) * S + (dt[t] * u[t].double())[:, None] * B[t]
            want[t] = ((S * Cm[t]).sum(1) + skip.double() * u[t].double()) * P.silu(z[t])
        left.append(S)
        at += n
    left = torch.stack(left)
    state = state0.clone().cuda()
    got = ops.selective_scan(u.cuda(), xz.cuda(), bc.cuda(), 1, 2 + N, dtl.cuda(), bias.cuda(), a_log.cuda(), skip.cuda(), state,
                             _step_context([0] * len(lengths), lengths)).double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.isnan(got[:, 4]).all() and torch.isnan(got).sum() == T
    assert torch.equal(torch.isnan(state.cpu()), torch.isnan(left))
    # 32-bit sums of up to 256 terms over up to 49 tokens, then one rounding to the type
    keep, tol = torch.arange(C) != 4, 1e-5 if dtype == torch.float32 else 4e-3
    assert (got - want)[:, keep].abs().max() < tol * float(want[:, keep].abs().max())
    assert (state.cpu().double() - left)[:, keep].abs().max() < 1e-5 * float(left[:, keep].abs().max())


@gpu
@pytest.mark.parametrize("C,N", [(2740, 9), (2740, 16), (1370, 32), (700, 64), (1370, 64), (1370, 100)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_selective_scan_of_many_channels(dtype, C, N):
    """Channels enough that a lane holds two or four states, to the same bounds."""
    test_selective_scan_alone(dtype, C, N)


@gpu
def test_selective_scan_at_the_ends_of_its_step_sizes_and_gates():
    """Step sizes and gates around where the kernel's own softplus and silu hand over to the library, and what is no finite number."""
    from palm_infra_amd.kernels import ops
    ends = torch.tensor([0.0, -0.0, 1e-3, -1e-3, 1.0, -1.0, 20.0, 20.1, 86.9, -86.9, 87.1, -87.1, 200.0, -200.0, float("inf"), -float("inf"), float("nan")])
    C, N, T = len(ends), 5, 33
    g = torch.Generator().manual_seed(3)
    u, bc, a_log = torch.randn(T, C, generator=g), torch.randn(T, 2 * N, generator=g), torch.zeros(C, N)
    for gates in (False, True):
        dtl, z = (torch.randn(T, C, generator=g), ends.repeat(T, 1)) if gates else (ends.repeat(T, 1), torch.randn(T, C, generator=g))
        dt, S, want = torch.nn.functional.softplus(dtl.double(), threshold=1e9), torch.zeros(C, N, dtype=P.F64), []
        dt = torch.where(dtl > 500, dtl.double(), dt)
        for t in range(T):
            S = torch.exp(-dt[t][:, None]) * S + (dt[t] * u[t].double())[:, None] * bc[t, :N].double()
            want.append((S * bc[t, N:].double()).sum(1) * z[t].double() / (1 + torch.exp(-z[t].double())))
        want, state = torch.stack(want), torch.zeros(1, C, N).cuda()
        got = ops.selective_scan(u.cuda(), torch.cat([u, z], 1).cuda(), bc.cuda(), 0, N, dtl.cuda(), torch.zeros(C).cuda(), a_log.cuda(),
                                 torch.zeros(C).cuda(), state, _step_context([0], [T])).double().cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        # each channel against its own size: sums of 32-bit terms over 33 tokens (and below 2^-126 nothing is compared)
        keep = torch.isfinite(want)
        size = torch.where(keep, want, 0.0).abs().amax(0)
        assert (torch.where(keep, got - want, 0.0).abs().amax(0) <= 1e-5 * size + 1e-37).all()


@gpu
def test_selective_scan_softplus_and_silu_to_the_last_places():
    """One token from an empty state with inputs of one is softplus(step) times silu(gate): both within some halves of the last place of
    64 bits, between the points where the library's functions take over."""
    from palm_infra_amd.kernels import ops
    small = torch.logspace(-7, 0, 500)
    x = torch.cat([torch.linspace(-86.9, 86.9, 6001), small, -small])
    C, one = len(x), torch.ones(1, len(x))
    for gates in (False, True):
        dtl, z = (one, x[None]) if gates else (x[None], one)
        got = ops.selective_scan(one.cuda(), torch.cat([one, z], 1).cuda(), torch.ones(1, 2).cuda(), 0, 1, dtl.contiguous().cuda(), torch.zeros(C).cuda(),
                                 torch.zeros(C, 1).cuda(), torch.zeros(C).cuda(), torch.zeros(1, C, 1).cuda(), _step_context([0], [1])).double().cpu()[0]
        step, gate = dtl[0].double(), z[0].double()
        want = (step.clamp(min=0) + torch.log1p(torch.exp(-step.abs()))) * gate / (1 + torch.exp(-gate))
        # 2.3 and 3.1 halves of a place (2^-24) were measured for the two functions over all such arguments, one more is the last product's
        worst = float(((got - want) / want).abs().max()) * 2 ** 24
        assert worst <= 2.3 + 3.1 + 1 + 0.5, (gates, worst)


@gpu
@pytest.mark.parametrize("dk,dv", [(12, 28), (40, 72)])      # the second pair is one that the matrix-core kernel takes in bfloat16
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_differential_attention_kernel_far_keys_page_borders_and_the_causal_edge(dtype, dk, dv):
    """Keys made so that one decides a query's output: far back, on either side of a page border, at the query's own
    position; and a large aligned key one position after the query, which the query must not see.  Whole, and with
    the last tokens one by one; two sequences of unequal lengths in one batch."""
    from palm_infra_amd.cache import KVNeed, ModelCache
    from palm_infra_amd.kernels import ops
    from palm_infra_amd.parts import make_context
    torch.manual_seed(3)
    H, G = 4, 2
    scale, lam, gain, eps = 0.5, 0.4, 0.6, 1e-6
    assert ops.diff_mfma_serves(torch.empty(0, dtype=dtype), dk, dv) == (dtype == torch.bfloat16 and dk == 40)
    T = [330, 71]
    width = 2 * (H + G) * dk + G * dv
    seqs = [torch.randn(t, width) * 0.5 for t in T]
    direction = torch.randn(dk)
    direction /= direction.norm()

    def aim(rows, query, key, head=1, which=0):
        g = head // (H // G)
        rows[query, (head * 2 + which) * dk:(head * 2 + which + 1) * dk] = direction * 9.0
        rows[key, 2 * H * dk + (g * 2 + which) * dk:2 * H * dk + (g * 2 + which + 1) * dk] = direction * 9.0

    # (query, key): far, page borders, own position; the key after query 200 must stay unseen
    for qy, ky in ((329, 2), (300, 63), (310, 64), (127, 127), (128, 127), (192, 128), (65, 0)):
        aim(seqs[0], qy, ky)
    aim(seqs[0], 200, 201, which=1)
    aim(seqs[1], 70, 64)
    aim(seqs[1], 63, 1, head=2, which=1)
    q_w, k_w = torch.rand(dk) + 0.5, torch.rand(dk) + 0.5
    seqs = [s.to(dtype) for s in seqs]

    def plain(rows):
        r = rows.double()
        n = r.shape[0]
        q = P.rms_norm(r[:, :2 * H * dk].view(n, H, 2, dk), q_w.double(), eps)
        k = P.rms_norm(r[:, 2 * H * dk:2 * (H + G) * dk].view(n, G, 2, dk), k_w.double(), eps)
        if dtype == torch.bfloat16:                                # the kernel keeps normed q and k in the run's type
            q, k = q.bfloat16().double(), k.bfloat16().double()
        v = r[:, 2 * (H + G) * dk:].view(n, G, dv)
        causal = torch.tril(torch.ones(n, n, dtype=torch.bool))
        out = torch.zeros(n, H, dv, dtype=P.F64)
        for hd in range(H):
            g = hd // (H // G)
            a = [torch.softmax(((q[:, hd, j] @ k[:, g, j].T) * scale).masked_fill(~causal, -math.inf), -1) @ v[:, g] for j in range(2)]
            out[:, hd] = P.unit_rms(a[0] - lam * a[1], eps) * gain
        return out.reshape(n, H * dv)

    want = [plain(s) for s in seqs]
    tol = 2e-5 if dtype == torch.float32 else 4e-2
    need = KVNeed(2 * G, dk, None, value_heads=G, value_dim=dv)
    cache = ModelCache([[need]], [None], 64 * 12, 4, None, dtype, torch.device("cuda"))
    lc = cache.layer_caches[0]
    for tail in (0, 9):
        slots = [cache.open() for _ in T]
        got = [[] for _ in T]
        steps = [[(b, 0, t - tail) for b, t in enumerate(T)]] + [[(b, t - tail + i, 1) for b, t in enumerate(T)] for i in range(tail)]
        for step in steps:
            growth = [(slots[b], n) for b, _, n in step]
            cache.reserve(growth)
            ctx = make_context([slots[b] for b, _, _ in step], [lo for _, lo, _ in step], [[0] * n for _, _, n in step], dtype, "cuda")
            rows = torch.cat([seqs[b][lo:lo + n] for b, lo, n in step]).cuda()
            q = ops.diff_qkv_store(rows, H, G, dk, dv, q_w.cuda(), k_w.cuda(), eps, lc.k, lc.v, lc.kv.table_dev, ctx)
            o = ops.attention_diff(q, lc.k, lc.v, lc.kv.table_dev, ctx, H, G, dk, dv, scale, lam, gain, eps).double().cpu()
            cache.commit(growth)
            at = 0
            for b, _, n in step:
                got[b].append(o[at:at + n])
                at += n
        for b in range(len(T)):
            err = (torch.cat(got[b]) - want[b]).abs().max()
            assert err < tol, f"sequence {b}, last {tail} one by one: {err}"
        for s in slots:
            cache.close(s)
    cache.check()


@gpu
@pytest.mark.parametrize("heads,kv_heads,dk,dv", [(4, 1, 64, 128), (8, 2, 128, 256), (6, 3, 40, 72), (3, 3, 96, 64), (8, 2, 256, 256), (4, 1, 32, 20)])
@pytest.mark.parametrize("lengths", [(1, 15), (16, 17, 64), (65, 129, 33), (700, 300, 513, 64)])
def test_differential_attention_of_prompts_at_the_edges_of_its_blocks(heads, kv_heads, dk, dv, lengths):
    """Prompts on the matrix cores in blocks of four waves (one or two pages in LDS, heads of a block that share keys or do not) against
    64 bits, over pages whose places beyond the sequences hold NaN, and with keys already there."""
    check_differential_prompts(heads, kv_heads, dk, dv, lengths, waves=4)


@gpu
@pytest.mark.parametrize("heads,kv_heads,dk,dv,lengths,waves", [
    (16, 4, 128, 256, (1100, 1037, 63), 8), (16, 4, 128, 256, (2048, 17), 8), (16, 4, 128, 256, (1000,), 4),          # one page of either kind in LDS
    (16, 4, 64, 128, (1100, 1037, 63, 700), 8), (16, 4, 64, 128, (1100, 1037, 63), 4), (8, 2, 40, 72, (513,) * 16, 8),
    (12, 6, 64, 128, (1100, 1037, 63, 700, 129), 8), (12, 12, 96, 64, (1100, 1037, 63, 700, 129), 8)])                # two heads a block, and one
def test_differential_attention_of_prompts_in_blocks_of_eight_waves(heads, kv_heads, dk, dv, lengths, waves):
    """Prompts on both sides of where the blocks of eight waves begin: heads and runs of queries that they share a page for, ends of
    sequences inside a block, waves without a query."""
    check_differential_prompts(heads, kv_heads, dk, dv, lengths, waves)


def check_differential_prompts(heads, kv_heads, dk, dv, lengths, waves):
    from palm_infra_amd.kernels import ops
    assert ops.attention_diff_lib(dk, dv).palm_attention_diff_mfma_waves(len(lengths), max(lengths), heads, kv_heads) == waves
    torch.manual_seed(sum(lengths) + dk)
    scale, lam, gain, eps = dk ** -0.5, 0.4, 0.6, 1e-6
    starts = [70 * (b % 2) for b in range(len(lengths))]
    ends = [s + n for s, n in zip(starts, lengths)]
    pages = [(e + 63) // 64 for e in ends]
    table = torch.zeros(len(lengths), max(pages), dtype=torch.int32)
    order = torch.randperm(sum(pages)).int()
    for b, n in enumerate(pages):
        table[b, :n] = order[sum(pages[:b]):sum(pages[:b + 1])]
    k_cache = torch.full((sum(pages), 2 * kv_heads, 64, dk), math.nan).bfloat16()
    v_cache = torch.full((sum(pages), kv_heads, dv, 64), math.nan).bfloat16()
    q = torch.randn(sum(lengths), heads, 2, dk).bfloat16()
    want, at = [], 0
    for b, end in enumerate(ends):
        k, v = (torch.randn(end, 2 * kv_heads, dk) * 2).bfloat16(), torch.randn(end, kv_heads, dv).bfloat16()
        for p in range(pages[b]):
            here = slice(64 * p, min(end, 64 * p + 64))
            k_cache[table[b, p], :, :here.stop - here.start] = k[here].transpose(0, 1)
            v_cache[table[b, p], :, :, :here.stop - here.start] = v[here].permute(1, 2, 0)
        mine = q[at:at + lengths[b]].double()
        at += lengths[b]
        hidden = torch.arange(end) > starts[b] + torch.arange(lengths[b])[:, None]
        out = torch.empty(lengths[b], heads, dv, dtype=P.F64)
        for h in range(heads):
            g = h // (heads // kv_heads)
            a = [torch.softmax((mine[:, h, m] @ k[:, 2 * g + m].double().T * scale).masked_fill(hidden, -math.inf), -1) @ v[:, g].double() for m in range(2)]
            out[:, h] = P.unit_rms(a[0] - lam * a[1], eps) * gain
        want.append(out.reshape(lengths[b], -1))
    cum = [0]
    for n in lengths:
        cum.append(cum[-1] + n)
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")

    class Ctx:
        seq_slot, seq_start, seq_new, cu_new = ints(list(range(len(lengths)))), ints(starts), ints(list(lengths)), ints(cum)
        n_tokens, n_seqs, max_new, is_decode = cum[-1], len(lengths), max(lengths), False

    got = ops.attention_diff_mfma(q.view(cum[-1], -1).cuda(), k_cache.cuda(), v_cache.cuda(), table.cuda(), Ctx, heads, kv_heads, dk, dv, scale, lam, gain, eps)
    # a weight is rounded to bfloat16 once (2^-9 of it), the result once more, and a1 - lambda a2 is shorter than its terms
    err = (got.double().cpu() - torch.cat(want)).norm() / torch.cat(want).norm()
    assert err < 6e-3, f"{err}"
    assert (got.double().cpu() - torch.cat(want)).abs().max() < 0.1 * float(torch.cat(want).abs().max())


# ---- whole models ----------------------------------------------------------------------------------------

@gpu
@pytest.mark.parametrize("name,dtype", CASES)
def test_each_request_alone_and_whole(tmp_path_factory, name, dtype):
    from palm_infra_amd.engine import StepEntry
    eng = engine_for(tmp_path_factory, name, dtype)
    for ids in S.prompts(raw_of(name), LENGTHS[name]):
        slot = eng.open()
        got = eng.step([StepEntry(slot, ids, list(range(len(ids))))])
        eng.close(slot)
        assert_close(got, reference(tmp_path_factory, name, dtype, ids), dtype, f"{name} whole {len(ids)}")
    eng.cache.check()


@gpu
@pytest.mark.parametrize("name,dtype", CASES)
def test_prompt_then_every_token_alone_from_the_first(tmp_path_factory, name, dtype):
    """Token-by-token decoding from the very first token (every state starts from zero, the convolution from its
    zero padding), through recorded steps, across page borders; against the whole prompt in one step."""
    from palm_infra_amd.engine import StepEntry
    eng = engine_for(tmp_path_factory, name, dtype)
    ids = S.prompts(raw_of(name), [150], seed=4)[0]
    ref = reference(tmp_path_factory, name, dtype, ids)
    slot = eng.open()
    pool = Pool(dtype, f"{name} one by one")
    for t, tok in enumerate(ids):
        pool.add(eng.step([StepEntry(slot, [tok], [0])]), ref[t:t + 1])
        assert eng.length(slot) == t + 1
    eng.close(slot)
    pool.check()


@gpu
@pytest.mark.parametrize("name,dtype", CASES)
@pytest.mark.parametrize("portion", [2, 3, 7, 64, 65])
def test_prompt_in_portions(tmp_path_factory, name, dtype, portion):
    from palm_infra_amd.engine import StepEntry
    eng = engine_for(tmp_path_factory, name, dtype)
    ids = S.prompts(raw_of(name), [140], seed=5)[0]
    ref = reference(tmp_path_factory, name, dtype, ids)
    slot = eng.open()
    got = []
    for lo in range(0, len(ids), portion):
        piece = ids[lo:lo + portion]
        got.append(eng.step([StepEntry(slot, piece, list(range(len(piece))))]))
    eng.close(slot)
    assert_close(torch.cat(got), ref, dtype, f"{name} in portions of {portion}")


@gpu
@pytest.mark.parametrize("name,dtype", CASES)
def test_batches_of_unequal_requests_and_reused_slots(tmp_path_factory, name, dtype):
    """Two batches through the same slots and pages: prompts of unequal lengths in one step minus their last tokens,
    which come one a step; a request that has no tokens left ends and gives its slot and pages back at once."""
    from palm_infra_amd.cache import KVNeed
    from palm_infra_amd.engine import StepEntry
    eng = engine_for(tmp_path_factory, name, dtype)
    paged = eng.cache.groups_of(KVNeed)
    for round_no, (seed, tails) in enumerate([(6, [0, 1, 9, 3, 20, 5, 2, 11]), (7, [12, 0, 2, 7, 30, 1, 1, 4])]):
        lengths = LENGTHS[name] if round_no == 0 else LENGTHS[name][::-1]
        reqs = S.prompts(raw_of(name), lengths, seed=seed)
        tails = [min(t, len(r) - 1) for t, r in zip(tails, reqs)]
        slots = [eng.open() for _ in reqs]
        assert sorted(slots) == list(range(len(reqs)))                # the second batch gets the first one's slots
        cuts = [len(r) - t for r, t in zip(reqs, tails)]
        got = {i: [] for i in range(len(reqs))}
        out = eng.step([StepEntry(s, r[:c], list(range(c))) for s, r, c in zip(slots, reqs, cuts)])
        o = 0
        for i, c in enumerate(cuts):
            got[i].append(out[o:o + c])
            o += c
        live, fed = list(range(len(reqs))), list(cuts)
        while True:
            for i in [i for i in live if fed[i] == len(reqs[i])]:
                eng.close(slots[i])
                live.remove(i)
            if not live:
                break
            out = eng.step([StepEntry(slots[i], [reqs[i][fed[i]]], [0]) for i in live])
            for r, i in enumerate(live):
                got[i].append(out[r:r + 1])
                fed[i] += 1
        for i, r in enumerate(reqs):
            assert_close(torch.cat(got[i]), reference(tmp_path_factory, name, dtype, r), dtype,
                                     f"{name} batch {round_no} request {i} ({len(r)} tokens, {tails[i]} one by one)")
        eng.cache.check()
        assert all(g.table.pages.held_count == 0 for g in paged)


@gpu
@pytest.mark.parametrize("name,dtype", [("P", "float32"), ("Q", "bfloat16"), ("Q", "float32")])
def test_long_decoding(tmp_path_factory, name, dtype):
    """A short prompt, then some hundred tokens one by one over several pages, two sequences side by side that
    started at different lengths."""
    from palm_infra_amd.engine import StepEntry
    eng = engine_for(tmp_path_factory, name, dtype)
    a, b = S.prompts(raw_of(name), [330, 270], seed=8)
    refs = [reference(tmp_path_factory, name, dtype, a), reference(tmp_path_factory, name, dtype, b)]
    sa, sb = eng.open(), eng.open()
    first = eng.step([StepEntry(sa, a[:70], [69]), StepEntry(sb, b[:10], [9])])
    pool = Pool(dtype, f"{name} long decoding")
    pool.add(first, torch.stack([refs[0][69], refs[1][9]]))
    for i in range(260):
        out = eng.step([StepEntry(sa, [a[70 + i]], [0]), StepEntry(sb, [b[10 + i]], [0])])
        pool.add(out, torch.stack([refs[0][70 + i], refs[1][10 + i]]))
    eng.close(sa)
    eng.close(sb)
    pool.check()


@gpu
@pytest.mark.parametrize("name", ["P", "Q"])
def test_recorded_and_launched_steps_agree(tmp_path_factory, name):
    """Decode steps replayed from a HIP graph against the same steps launched kernel by kernel, several replays with
    other work between them."""
    from palm_infra_amd.engine import StepEntry
    ids = S.prompts(raw_of(name), [90], seed=9)[0]
    outs = []
    for graphs in (True, False):
        eng = engine_for(tmp_path_factory, name, "float32", graphs=graphs)
        slot = eng.open()
        got = [eng.step([StepEntry(slot, ids[:50], [49])])]
        for t in range(50, 90):
            got.append(eng.step([StepEntry(slot, [ids[t]], [0])]))
            torch.cuda.synchronize()
        eng.close(slot)
        outs.append(torch.cat(got).cpu())
    assert torch.allclose(outs[0], outs[1], atol=1e-5)
    assert_close(outs[0], reference(tmp_path_factory, name, "float32", ids)[49:], "float32", f"{name} recorded steps")


@gpu
@pytest.mark.parametrize("name", ["P", "Q", "R"])
def test_greedy_generation_through_generate(tmp_path_factory, name):
    from palm_infra_amd.sampling import GREEDY
    eng = engine_for(tmp_path_factory, name, "float32")
    cfg, w = P.read_model(model_dir(tmp_path_factory, name, "float32"))
    prompts = S.prompts(raw_of(name), [5, 1, 66, 19], seed=10)
    results, metrics = eng.generate(prompts, GREEDY, max_new_tokens=12, ignore_eos=True, max_batch=3)
    for p, r in zip(prompts, results):
        assert r.token_ids == P.greedy(cfg, w, p, 12), f"{name}: prompt of {len(p)} tokens"
    eng.cache.check()
    assert eng.cache.slots.held_count == 0


@gpu
def test_command_line_generates_for_the_design(tmp_path_factory, capsys):
    from palm_infra_amd.engine.cli import chat_main
    d = model_dir(tmp_path_factory, "R", "float32")
    cfg, w = P.read_model(d)
    rc = chat_main(["--package", str(d), "--prompt-ids", "5,6,7", "--max-new-tokens", "6", "--temperature", "0",
                    "--dtype", "float32", "--ignore-eos"])
    assert rc == 0
    assert " ".join(str(t) for t in P.greedy(cfg, w, [5, 6, 7], 6)) in capsys.readouterr().out


@gpu
def test_trace_replay_of_many_short_requests_counted_by_their_tokens(tmp_path_factory, tmp_path):
    """bin/trace_run as a child process: six requests of 70 tokens in one batch and then one token each, with
    --max-tokens counting the tokens they hold (426) and not the pages they touch (twelve)."""
    import json
    import subprocess
    import sys
    from pathlib import Path
    import numpy as np
    d = model_dir(tmp_path_factory, "P", "float32")
    reqs = S.prompts(raw_of("P"), [71] * 6, seed=11)
    steps = [{"step": 0, "entries": [{"id": f"r{i}", "tokens": r[:70], "want": [0, 69]} for i, r in enumerate(reqs)], "end": []},
             {"step": 1, "entries": [{"id": f"r{i}", "tokens": r[70:], "want": [0]} for i, r in enumerate(reqs)], "end": [f"r{i}" for i in range(6)]}]
    root = Path(__file__).resolve().parent.parent
    proc = subprocess.run([sys.executable, str(root / "bin" / "trace_run"), "--model", str(d), "--dtype", "float32", "--out", str(tmp_path / "o"),
                           "--max-tokens", "426"], input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stderr[-2000:]
    assert [line for line in proc.stdout.splitlines() if line.startswith("done")] == ["done 0", "done 1"]
    V = raw_of("P")["vocab"]
    first = torch.from_numpy(np.fromfile(tmp_path / "o" / "0.f32", dtype="<f4").reshape(-1, V).copy())
    second = torch.from_numpy(np.fromfile(tmp_path / "o" / "1.f32", dtype="<f4").reshape(-1, V).copy())
    for i, r in enumerate(reqs):
        ref = reference(tmp_path_factory, "P", "float32", r)
        assert_close(first[2 * i:2 * i + 2], ref[[0, 69]], "float32", f"request {i}, prompt")
        assert_close(second[i:i + 1], ref[70:71], "float32", f"request {i}, decoded")
