"""Linear attention and its forms over chunks that hold resets, which are worked in one unit with the episodes kept apart by masks:
every place of an episode's boundary in a chunk against the oracle, and the screen -- an episode with values beyond its bounds, or not finite, sends
the chunk to the units per episode, and the other episodes keep their bits."""
import numpy as np
import pytest
import torch

from gpu_util import TOL_BF16, TOL_F32, bf16_round, dev, relerr
from oracle import grad as G

pytestmark = pytest.mark.gpu

FORMS = ("plain", "gated", "normalised")


def _patterns(B, T, C):
    """Reset masks by where they lie in chunks of C rows."""
    def at(*ts):
        d = np.zeros((B, T), bool)
        d[:, [t for t in ts if t < T]] = True
        return d
    out = {"first_row": at(*range(0, T, C)), "last_row": at(*range(C - 1, T, C)), "every_row": np.ones((B, T), bool),
           "tile_edges": at(15, 16, C + 15, C + 17, T - 1), "runs": at(5, 6, 7, C + 8, C + 9, 2 * C - 1, 2 * C)}
    out["one_sequence_only"] = at(3, C + 20)
    out["one_sequence_only"][1:] = False
    return out


def _case(B, T, H, d, dtype, seed):
    rng = np.random.default_rng(seed)
    x = {n: (rng.standard_normal((B, T, H, d)) / 8).astype(np.float32) for n in ("q", "k", "v", "do")}
    if dtype == "bf16":
        x = {n: bf16_round(a) for n, a in x.items()}
    x["g"] = (-0.2 * np.abs(rng.standard_normal((B, T, H)))).astype(np.float32)
    x["S0"] = (rng.standard_normal((B, H, d, d)) * 0.1).astype(np.float32)
    x["z0"] = np.abs(rng.standard_normal((B, H, d))).astype(np.float32)
    return x


def _run(form, x, done, dtype):
    from memorax_amd import functional as Fn
    td = torch.bfloat16 if dtype == "bf16" else torch.float32
    q, k, v = (dev(x[n], td).requires_grad_() for n in ("q", "k", "v"))
    ins, S0, dn = [q, k, v], dev(x["S0"]).requires_grad_(), dev(done)
    if form == "plain":
        out = Fn.linear_attention(q, k, v, dn, S0, "elu1")
    elif form == "gated":
        ins.append(dev(x["g"]).requires_grad_())
        out = Fn.gated_linear_attention(*ins, dn, S0, "elu1")
    else:
        ins.append(dev(x["z0"]).requires_grad_())
        out = Fn.normalised_linear_attention(q, k, v, dn, S0, ins[3], "elu1")
    grads = torch.autograd.grad(out[0], ins + [S0], dev(x["do"], td))
    torch.cuda.synchronize()
    names = ["dq", "dk", "dv"] + {"plain": [], "gated": ["dg"], "normalised": ["dz0"]}[form] + ["dS0"]
    return dict(zip(["o", "S_last", "z_last"], out), **dict(zip(names, grads)))


def _oracle(form, x, done, stored):
    a = (x["q"], x["k"], x["v"])
    if form == "plain":
        return G.linear_attention_grads(*a, done, x["S0"], x["do"], None, "elu1")
    if form == "gated":
        return G.gated_linear_attention_grads(*a, x["g"], done, x["S0"], x["do"], None, "elu1")
    # the backward's quotients are those that were stored
    ref = G.normalised_linear_attention_grads(*a, done, x["S0"], x["z0"], x["do"], o_stored=stored.detach().float().cpu().numpy())
    return dict(ref, o=G.normalised_linear_attention_grads(*a, done, x["S0"], x["z0"], x["do"])["o"])


@pytest.mark.parametrize("d", [64, 48, 32])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("form", FORMS)
def test_episode_boundaries_anywhere_in_a_chunk(form, dtype, d):
    C = 64 if dtype == "bf16" else 32
    tol = TOL_BF16 if dtype == "bf16" else TOL_F32
    for T in (2 * C + 9, C - 3):
        for name, done in _patterns(2, T, C).items():
            print(f"case one_unit form={form} dtype={dtype} d={d} T={T} pattern={name}", flush=True)
            x = _case(2, T, 2, d, dtype, T + d)
            got = _run(form, x, done, dtype)
            ref = _oracle(form, x, done, got["o"])
            for n, r in ref.items():
                if n not in got:
                    continue
                # Two gradients are differences and held to their terms.  A log-decay's: q.dq and k.dk.  The normalised form's dq and dk where every row is
                # an episode (o = v whatever q and k): do.v / den phi(k), 64 products of 1/8 x 1/8 over a den of about 64, 2^-6.
                scale = max(np.abs(r).max(), 2.0**-6 if form == "normalised" and n in ("dq", "dk") else 1e-6)
                if n == "dg":
                    scale += np.abs((x["q"] * ref["dq"]).sum(-1)).max() + np.abs((x["k"] * ref["dk"]).sum(-1)).max()
                err = np.abs(got[n].detach().float().cpu().numpy() - r).max() / scale
                assert err <= (5 * tol if n == "dg" else tol), (name, n, err)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("what", [float("nan"), float("inf"), 2.0**21])
def test_an_episode_beyond_the_screen_stays_by_itself(form, dtype, what):
    C = 64 if dtype == "bf16" else 32
    T = 2 * C
    lo, hi = C + 10, C + 20
    done = np.zeros((1, T), bool)
    done[0, [lo, hi]] = True
    x = _case(1, T, 2, 64, dtype, 5)
    bad = {n: a.copy() for n, a in x.items()}
    for n in ("q", "k", "v", "do"):
        bad[n][0, lo + 2:hi - 1] = what
    print(f"case one_unit screen form={form} dtype={dtype} what={what}", flush=True)
    a, b = _run(form, x, done, dtype), _run(form, bad, done, dtype)
    keep = np.ones(T, bool)
    keep[lo:hi] = False
    for n in a:
        u, w = (t[:, keep] if t.dim() >= 3 and t.shape[1] == T else t for t in (a[n], b[n]))
        assert torch.equal(u, w), n


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("name", ["q", "k", "v", "do"])
def test_one_element_beyond_the_screen(form, dtype, name):
    """The screen sees what every lane of every wave holds, not the first lane's share of the chunk."""
    C = 64 if dtype == "bf16" else 32
    T, lo, hi = 2 * C, C + 10, C + 20
    done = np.zeros((1, T), bool)
    done[0, [lo, hi]] = True
    x = _case(1, T, 2, 64, dtype, 6)
    good = _run(form, x, done, dtype)
    keep = np.ones(T, bool)
    keep[lo:hi] = False
    for row, col in ((lo, 63), (lo + 3, 0), (lo + 4, 33), (hi - 1, 20)):
        bad = dict(x, **{name: x[name].copy()})
        bad[name][0, row, 1, col] = np.nan
        print(f"case one_unit element form={form} dtype={dtype} of={name} at={row},{col}", flush=True)
        got = _run(form, bad, done, dtype)
        for n in good:
            u, w = (t[:, keep] if t.dim() >= 3 and t.shape[1] == T else t for t in (good[n], got[n]))
            assert torch.equal(u, w), n


@pytest.mark.parametrize("chunks", [3, 12])   # a workgroup per sequence, a workgroup per chunk
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("form", FORMS)
def test_a_reset_on_a_chunk_s_first_row_drops_what_enters_it(form, dtype, chunks):
    """The episode that ends with a chunk leaves a state, and a sum of keys, that is not finite: no row of the next chunk is of that episode, and its
    inputs pass the screen."""
    C = 64 if dtype == "bf16" else 32
    T = chunks * C
    done = np.zeros((1, T), bool)
    done[0, [C, 2 * C + 7]] = True
    x = _case(1, T, 2, 64, dtype, 7)
    print(f"case one_unit first row form={form} dtype={dtype} chunks={chunks}", flush=True)
    good = _run(form, x, done, dtype)
    for what in (float("nan"), float("inf")):
        bad = {n: a.copy() for n, a in x.items()}
        bad["k"][0, C - 5, 0, 11] = what
        got = _run(form, bad, done, dtype)
        for n in good:
            u, w = (t[:, C:] if t.dim() >= 3 and t.shape[1] == T else t for t in (good[n], got[n]))
            if n not in ("dS0", "dz0"):   # of the episode that enters the sequence
                assert torch.equal(u, w), n


@pytest.mark.parametrize("chunks", [4, 12])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("form", FORMS)
def test_a_reset_drops_what_comes_back_from_later_chunks(form, dtype, chunks):
    """The gradient of the state that leaves a chunk is not finite, the chunk's own rows pass the screen: it reaches the chunk's last episode and no other."""
    C = 64 if dtype == "bf16" else 32
    T = chunks * C
    done = np.zeros((1, T), bool)
    done[0, [C, 2 * C + 7]] = True
    x = _case(1, T, 2, 64, dtype, 8)
    print(f"case one_unit later chunk form={form} dtype={dtype} chunks={chunks}", flush=True)
    good = _run(form, x, done, dtype)
    for what in (float("nan"), float("inf")):
        bad = dict(x, do=x["do"].copy())
        bad["do"][0, 3 * C + 3, 1, 40] = what
        got = _run(form, bad, done, dtype)
        for n in good:
            u, w = (t[:, :2 * C + 7] if t.dim() >= 3 and t.shape[1] == T else t for t in (good[n], got[n]))
            assert torch.equal(u, w), n


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("what", [float("nan"), float("inf"), 200.0])
def test_a_gate_beyond_bounds_stays_in_its_episode(what, dtype):
    """Gates are not screened: what they make of a step's decay meets the rows of its own episode only."""
    C = 64 if dtype == "bf16" else 32
    T, lo, hi = 3 * C, C + 10, C + 20
    done = np.zeros((1, T), bool)
    done[0, [5, lo, hi, 2 * C]] = True
    x = _case(1, T, 2, 64, dtype, 9)
    good = _run("gated", x, done, dtype)
    keep = np.ones(T, bool)
    keep[lo:hi] = False
    for row in (lo + 1, lo + 4, hi - 1):
        bad = dict(x, g=x["g"].copy())
        bad["g"][0, row, 1] = what
        print(f"case one_unit gate dtype={dtype} what={what} row={row}", flush=True)
        got = _run("gated", bad, done, dtype)
        for n in good:
            u, w = (t[:, keep] if t.dim() >= 3 and t.shape[1] == T else t for t in (good[n], got[n]))
            assert torch.equal(u, w), n
