"""Performance cases of the framework: dump intervals of lattice ensembles.

A pass is what a run does between two rows of its entropy file: advance every
chain by a batch of Yoshida-6 steps, then the linear-mode energies and both
entropies (``Ensemble.batch``, or ``move`` + ``linenergies`` for a program that
issues them one by one; with ``check`` also the total energy of every chain,
the usual watch on the integrator).  The ensemble stays on the GPU from pass to
pass, as in a run; a pass returns the energies, the entropies and the state.

``prepare`` makes the initial state on the GPU from the seed (running waves
with random phases: most of the energy in the lowest modes, the rest of the
spectrum weakly excited) and creates the ensemble; ``exact`` integrates the
same state with plain torch operations in FP64.
"""
import ctypes
import math

import numpy as np
import torch

import nlchains_amd as nlc

# FLOP per site-step (FMA = 2, exp and sincos = 0); DNLS: 7 x (two complex FFTs
# of 5 n log2 n plus 16 pointwise)
_FLOP = {"DNKG": 70, "dDNKG": 70, "FPUT": 119, "Toda": 56}

_DEFAULTS = {"form": "batch", "precision": "fp64", "m": 0.0, "alpha": 0.0, "beta": 0.0, "check": False}


def _case(name, **kw):
    return {"name": name, **_DEFAULTS, **kw}


def listed():
    return [
        # the smallest runs: short FPUT-beta chains, a batch of tens of
        # microseconds where launches and latency count
        _case("fput_64x1024", model="FPUT", n=64, copies=1024, steps=100, dt=0.1, beta=1.0),
        # the usual large ensemble of the real models (DNKG, 1024 sites x 16384)
        _case("dnkg_1024x16384", model="DNKG", n=1024, copies=16384, steps=100, dt=0.05, m=1.0, beta=1.0),
        # FPUT-alpha at an odd length, issued as move + linenergies
        _case("fput_alpha_1001x4096", model="FPUT", n=1001, copies=4096, steps=100, dt=0.05, alpha=0.25,
              form="move"),
        # FPUT alpha + beta chains longer than a wavefront holds
        _case("fput_4096x1024", model="FPUT", n=4096, copies=1024, steps=100, dt=0.05, alpha=0.25, beta=0.5),
        # few long chains, beyond a workgroup's registers
        _case("dnkg_20000x256", model="DNKG", n=20000, copies=256, steps=100, dt=0.05, m=1.0, beta=1.0),
        # Toda chains of many lengths in one context (thermalisation against
        # size), with the energy of every chain
        _case("toda_ragged_8192", model="Toda", n=2048, n_lo=32, copies=8192, steps=100, dt=0.05, alpha=1.0,
              check=True),
        # disordered DNKG: energies are a projection on the eigenvectors
        _case("ddnkg_512x8192", model="dDNKG", n=512, copies=8192, steps=100, dt=0.05, beta=1.0),
        # DNLS at its usual size, the longest passes; the same in FP32C
        _case("dnls_4096x4096", model="DNLS", n=4096, copies=4096, steps=40, dt=0.01, beta=1.0),
        _case("dnls_fp32c_4096x2048", model="DNLS", n=4096, copies=2048, steps=20, dt=0.01, beta=1.0,
              precision="fp32c"),
        # DNLS at shorter, not power-of-two and long chain lengths
        _case("dnls_1024x4096", model="DNLS", n=1024, copies=4096, steps=20, dt=0.01, beta=1.0),
        _case("dnls_1000x2048", model="DNLS", n=1000, copies=2048, steps=20, dt=0.01, beta=1.0),
        _case("dnls_16384x256", model="DNLS", n=16384, copies=256, steps=20, dt=0.01, beta=1.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n):
    """Whether the prime factors of n are 2, 3, 5 and 7."""
    for f in (2, 3, 5, 7):
        while n % f == 0:
            n //= f
    return n == 1


def _draw_length(rng, lo, hi):
    """A chain length, log-uniform: powers of two, round (smooth) lengths and any others, a third each."""
    n, kind = _log_int(rng, lo, hi), rng.randrange(3)
    if kind == 0:
        return 1 << min(max(round(math.log2(n)), math.ceil(math.log2(lo))), int(math.log2(hi)))
    if kind == 1:
        while not _smooth(n):
            n -= 1
    return max(n, lo)


def draw(rng):
    """A dump interval of the ranges above: models, lengths of 16 to 32768 sites, ensembles of 2^15 to 2^24 sites."""
    what = rng.choice(["real", "real", "real", "dnls", "dnls", "ragged"])
    c = dict(_DEFAULTS, form=rng.choice(["batch", "batch", "move"]), check=rng.random() < 0.2)
    if what == "dnls":
        n = _draw_length(rng, 32, 32768)
        pow2 = n & (n - 1) == 0
        # an ensemble of awkward lengths is smaller: their transforms cost more
        sites = _log_int(rng, 1 << 15, 1 << (22 if pow2 else 21 if _smooth(n) else 19))
        c.update(model="DNLS", n=n, dt=0.01, beta=rng.choice([0.5, 1.0]), steps=_log_int(rng, 5, 20))
        if n == 4096 and rng.random() < 0.5:
            c.update(precision="fp32c")
    elif what == "ragged":
        sites = _log_int(rng, 1 << 16, 1 << 23)
        c.update(model=rng.choice(["Toda", "FPUT"]), n_lo=rng.choice([16, 32, 64]), n=rng.choice([512, 1024, 2048]),
                 dt=0.05, alpha=1.0, steps=_log_int(rng, 20, 100))
        if c["model"] == "FPUT":
            c.update(alpha=0.25, beta=0.5)
        c["copies"] = max(8, sites // (c["n"] // 3))
        return c
    else:
        model = rng.choice(["DNKG", "FPUT", "FPUT", "Toda", "dDNKG"])
        n = _draw_length(rng, 16, 600 if model == "dDNKG" else 32768)
        plain = n & (n - 1) == 0 or _smooth(n)
        sites = _log_int(rng, 1 << 16, 1 << (24 if plain or n < 128 else 21))
        c.update(model=model, n=n, dt=0.05, steps=_log_int(rng, 20, 200))
        if model == "DNKG":
            c.update(m=rng.choice([0.0, 0.5, 1.0]), beta=rng.choice([0.5, 1.0]))
        elif model == "dDNKG":
            c.update(beta=rng.choice([0.5, 1.0]))
        elif model == "Toda":
            c.update(alpha=rng.choice([0.5, 1.0]))
        else:
            a, b = rng.choice([(0.0, 1.0), (0.25, 0.0), (0.25, 0.5)])
            c.update(alpha=a, beta=b)
        if model in ("FPUT", "Toda") and n & (n - 1) == 0 and n <= 2048 and rng.random() < 0.2:
            c.update(precision="fp32c")
    c["copies"] = max(1, sites // c["n"])
    return c


# ---- inputs ---------------------------------------------------------------------


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _lengths(case):
    """Ragged ensembles: the length of every chain, powers of two from n_lo to n (the composition is the ensemble's
    own, not the seed's)."""
    choices = [1 << e for e in range(case["n_lo"].bit_length() - 1, case["n"].bit_length())]
    return np.random.default_rng(4).choice(np.array(choices, dtype=np.uint32), size=case["copies"])


def _masses(case):
    """dDNKG: the disorder is the model's own, not the seed's."""
    return np.random.default_rng(5).uniform(0.5, 1.5, size=case["n"])


def _waves(case, n, copies, gen):
    """copies x n x 2 doubles: random phases, mode amplitudes falling from the lowest n/8 modes to a weak background;
    energy density 0.1 (DNLS: norm density 1)."""
    dev = _device()
    k = torch.arange(n, device=dev, dtype=torch.float64)
    k = torch.minimum(k, n - k)
    amp = 1.0 / (1.0 + (8.0 * k / n) ** 4) + 0.02
    phase = torch.rand((copies, n), generator=gen, device=dev, dtype=torch.float64) * (2 * math.pi)
    if case["model"] == "DNLS":
        z = torch.fft.ifft(amp * torch.exp(1j * phase), dim=1) * (n / amp.square().sum().sqrt())
        return torch.view_as_real(z).contiguous()
    # q and p of independent phases; the amplitude of mode k over its frequency in q
    other = torch.rand((copies, n), generator=gen, device=dev, dtype=torch.float64) * (2 * math.pi)
    m = 1.0 if case["model"] in ("DNKG", "dDNKG") else 0.0
    w = torch.sqrt(m + 4 * torch.sin(math.pi * k / n) ** 2)
    if m == 0:
        amp = torch.where(k == 0, torch.zeros_like(amp), amp)
        w = torch.where(k == 0, torch.ones_like(w), w)
    scale = n / amp.square().sum().sqrt() * math.sqrt(0.2)
    q = torch.fft.ifft(amp / w * torch.exp(1j * phase), dim=1).real * scale
    p = torch.fft.ifft(amp * torch.exp(1j * other), dim=1).real * scale
    return torch.stack((q, p), dim=2).contiguous()


def _groups(case):
    """[(length, chain indices)] in ascending length."""
    if "n_lo" not in case:
        return [(case["n"], None)]
    lengths = _lengths(case)
    return [(int(n), np.flatnonzero(lengths == n)) for n in np.unique(lengths)]


def _initial(case, seed):
    """The initial chains of every length, in ascending length."""
    gen = torch.Generator(device=_device())
    gen.manual_seed(seed)
    return [_waves(case, n, case["copies"] if at is None else len(at), gen) for n, at in _groups(case)]


class _Shard:
    """The ensemble's own device memory as an array, in its device order."""

    def __init__(self, ens):
        ptr, size = ctypes.c_void_p(), ctypes.c_size_t()
        rc = nlc.lib.nlc_device_state(ens.handle, ctypes.byref(ptr), ctypes.byref(size))
        if rc:
            raise nlc.NlcError(rc, "nlc_device_state")
        self.ens = ens  # the memory is the ensemble's
        self.__cuda_array_interface__ = {"shape": (size.value // 8,), "typestr": "<f8", "data": (ptr.value, False),
                                         "version": 2}


def _precision(case):
    return nlc.FP32C if case["precision"] == "fp32c" else nlc.FP64


def prepare(case, seed):
    chains = _initial(case, seed)
    model = nlc.MODELS[case["model"]]
    force = dict(m=case["m"], alpha=case["alpha"], beta=case["beta"])
    if "n_lo" in case:
        ens = nlc.Ensemble.ragged(model, _lengths(case), case["dt"], precision=_precision(case), **force)
    else:
        masses = _masses(case) if case["model"] == "dDNKG" else None
        ens = nlc.Ensemble(model, case["n"], case["copies"], case["dt"], masses=masses, precision=_precision(case),
                           **force)
    # chains of one length are contiguous on the device, in ascending length
    # and otherwise in the caller's order
    shard = torch.as_tensor(_Shard(ens), device="cuda")
    at = 0
    for c in chains:
        shard[at:at + c.numel()].copy_(c.reshape(-1))
        at += c.numel()
    torch.cuda.synchronize()
    return {"ens": ens, "shard": shard, "steps": case["steps"], "form": case["form"], "check": case["check"]}


def run(state):
    ens = state["ens"]
    if state["form"] == "batch":
        energies, entropies = ens.batch(state["steps"])
    else:
        ens.move(state["steps"])
        energies, entropies = ens.linenergies()
    out = {"linenergies": energies, "entropies": entropies, "state": state["shard"]}
    if state["check"]:
        out["chain_energies"], _ = ens.chain_energies()
    return out


# ---- work -----------------------------------------------------------------------


def _flops(case, n, copies):
    sites = n * copies
    if case["model"] == "DNLS":
        step = 7 * (10 * math.log2(n) + 16)
    elif case["model"] == "FPUT" and case["alpha"] == 0:
        step = 91
    else:
        step = _FLOP[case["model"]]
    energy = 4 * n if case["model"] == "dDNKG" else 5 * math.log2(n)
    return sites * (step * case["steps"] + energy)


def work(case):
    # every site read and written once, the results written once
    if "n_lo" in case:
        sizes = [(n, len(at)) for n, at in _groups(case)]
    else:
        sizes = [(case["n"], case["copies"])]
    bytes_ = sum(32 * n * c + 8 * (n + 2) for n, c in sizes)
    if case["model"] == "dDNKG":
        bytes_ += 8 * case["n"] ** 2
    if case["check"]:
        bytes_ += 8 * case["copies"]
    return {"bytes": bytes_, "flops": sum(_flops(case, n, c) for n, c in sizes)}


# ---- the same in plain FP64 -------------------------------------------------------

# Yoshida (1990), 6th order, solution A: weights of the drifts and the kicks
_C = [0.392256805238780, 0.510043411918458, -0.471053385409757, 0.068753168252518,
      0.068753168252518, -0.471053385409757, 0.510043411918458, 0.392256805238780]
_D = [0.784513610477560, 0.235573213359357, -1.177679984178870, 1.315186320683906,
      -1.177679984178870, 0.235573213359357, 0.784513610477560]


def _move_real(case, q, p, masses):
    m, a, b, dt = case["m"], case["alpha"], case["beta"], case["dt"]

    def force():
        left, right = torch.roll(q, 1, 1), torch.roll(q, -1, 1)
        if case["model"] in ("DNKG", "dDNKG"):
            return left + right - q * ((masses if masses is not None else m) + 2 + b * q * q)
        dl, dr = q - left, right - q
        if case["model"] == "FPUT":
            return dr * (1 + dr * (a + b * dr)) - dl * (1 + dl * (a + b * dl))
        return (torch.exp(2 * a * dr) - torch.exp(2 * a * dl)) / (2 * a)

    for s in range(case["steps"]):
        for k in range(7):
            q += (2 if s and not k else 1) * _C[k] * dt * p
            p += _D[k] * dt * force()
    q += _C[7] * dt * p


def _move_dnls(case, z):
    n, dt = z.shape[1], case["dt"]
    k = torch.arange(n, device=z.device, dtype=torch.float64)
    w = 4 * torch.sin(math.pi * k / n) ** 2

    def turn(z, c):
        return z * torch.exp(-1j * (case["beta"] * dt * c) * (z.real.square() + z.imag.square()))

    for s in range(case["steps"]):
        for k in range(7):
            z = turn(z, (2 if s and not k else 1) * _C[k])
            z = torch.fft.ifft(torch.fft.fft(z, dim=1) * torch.exp(-1j * dt * _D[k] * w), dim=1)
    return turn(z, _C[7])


def _entropies(e, first):
    x = e[first:]
    norm = x.numel() / x.sum()
    y = norm * x
    return torch.stack((-torch.log(y).sum(), (y * torch.log(y)).sum()))


def _chain_energies(case, q, p, masses):
    m, a, b = case["m"], case["alpha"], case["beta"]
    d = torch.roll(q, -1, 1) - q
    h = 0.5 * p * p
    if case["model"] == "FPUT":
        h = h + 0.5 * d ** 2 + a * d ** 3 / 3 + 0.25 * b * d ** 4
    elif case["model"] == "Toda":
        h = h + (torch.exp(2 * a * d) - 1) / (4 * a * a) - d / (2 * a)
    else:
        h = h + 0.5 * d ** 2 + 0.5 * (masses if masses is not None else m) * q ** 2 + 0.25 * b * q ** 4
    return h.sum(dim=1)


def exact(case, seed):
    if work(case)["flops"] > 2e12:
        return None
    lin, ent, states, total = [], [], [], []
    for (n, at), c in zip(_groups(case), _initial(case, seed)):
        copies = c.shape[0]
        k = torch.arange(n, device=c.device, dtype=torch.float64)
        if case["model"] == "DNLS":
            z = _move_dnls(case, torch.view_as_complex(c))
            f = torch.fft.fft(z, dim=1)
            e = 4 * torch.sin(math.pi * k / n) ** 2 * (f.real.square() + f.imag.square()).sum(dim=0) / (n * copies)
            e[0] = 0
            first = 1
            a2 = z.real.square() + z.imag.square()
            d = torch.roll(z, -1, 1) - z
            total.append((d.real.square() + d.imag.square() + 0.5 * case["beta"] * a2 * a2).sum(dim=1))
            states.append(torch.view_as_real(z).reshape(-1))
        else:
            masses = torch.as_tensor(_masses(case), device=c.device) if case["model"] == "dDNKG" else None
            q, p = c[:, :, 0].clone(), c[:, :, 1].clone()
            _move_real(case, q, p, masses)
            if masses is not None:
                a = torch.diag(masses + 2)
                i = torch.arange(n, device=c.device)
                a[i, (i + 1) % n] -= 1
                a[(i + 1) % n, i] -= 1
                w2, v = torch.linalg.eigh(a.cpu())
                w2, v = w2.to(c.device), v.to(c.device)
                e = 0.5 / copies * (w2 * (q @ v).square() + (p @ v).square()).sum(dim=0)
                first = 0
            else:
                first = int(case["m"] == 0)
                w = torch.sqrt(case["m"] + 4 * torch.sin(math.pi * k / n) ** 2)
                g = torch.fft.fft(p, dim=1) - 1j * w * torch.fft.fft(q, dim=1)
                e = 0.5 / copies / n * (g.real.square() + g.imag.square()).sum(dim=0)
                if first:
                    e[0] = 0
            total.append(_chain_energies(case, q, p, masses))
            states.append(torch.stack((q, p), dim=2).reshape(-1))
        lin.append(e)
        ent.append(_entropies(e, first))
    out = {"linenergies": torch.cat(lin).cpu().numpy(), "entropies": torch.cat(ent).cpu().numpy(),
           "state": torch.cat(states)}
    if case["check"]:
        # the chains in the caller's order
        energies, everyone = np.empty(case["copies"]), np.arange(case["copies"])
        for (n, at), t in zip(_groups(case), total):
            energies[everyone if at is None else at] = t.cpu().numpy()
        out["chain_energies"] = energies
    return out
