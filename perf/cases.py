"""Timing cases of the (T) framework: what its users have it do.

A case is one call sequence through the public Python binding
(atrip_amd.hip.Context, atrip_amd.serve.Server) on a system of No occupied
and Nv virtual orbitals:

  run       E(T) (and E(cT)) over the tuple space or a range of it: the
            segment of one checkpoint or progress line, or the rest of a
            calculation resumed from a checkpoint
  tuples    per-tuple energies over a range
  batch     E(T) of many small systems in one call
  serve     a request loop over one context, from submission to the last result
  drop_in   host tensors in, E(T) out, everything released: one whole
            Atrip::run of a program that holds its tensors in host memory

Systems are the library's seeded synthetic ones (generated on the device) or,
for drop_in, host tensors drawn with the same distributions: orbital energies
uniform, amplitudes and integrals normal, T2 and V2 symmetric under the
exchange of both index pairs.  `exact` evaluates the same energies from the
closed-shell formulas with plain torch in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from atrip_amd import hip, serve

# bytes per element of the doubles operands of each form
OPERAND_BYTES = {"fp64": 8, "split_fp32": 6, "fp32": 4, "bf16x3": 6}
OPERAND_STORE = {"fp64": 0, "split_fp32": 1, "fp32": 2, "bf16x3": 3}


def n_tuples(nv):
    return nv * (nv + 1) * (nv + 2) // 6 - nv


def _case(kind, no, nv, precision="fp64", count=0, **more):
    c = {"kind": kind, "no": no, "nv": nv, "precision": precision,
         "count": count if 0 < count < n_tuples(nv) else 0,
         "at": 0.4, "with_j": False, "complex": False, "systems": 0}
    c.update(more)
    return c


def listed():
    return [
        # a water-sized molecule, the smallest whole calculation: latency
        # and launches
        dict(_case("run", 4, 36), name="water_fp64"),
        # a program that holds its tensors in host memory: upload, E(T),
        # release (the CPU-runnable configuration No=10, Nv=50)
        dict(_case("drop_in", 10, 50), name="drop_in_no10_nv50"),
        # a small molecule, whole calculation: the largest shape of the
        # batched workload on its own
        dict(_case("run", 16, 120), name="small_fp64"),
        # served mid-size shape, the segment between two progress lines
        dict(_case("run", 26, 308, count=200000), name="mid_fp64"),
        # the headline FP64 benchmark shape, the rest of a resumed calculation
        dict(_case("run", 40, 400, count=102000, at=1.0), name="large_fp64"),
        # split FP32 on an odd served shape (No = 31: every tile ragged)
        dict(_case("run", 31, 270, "split_fp32", count=200000), name="mid_split_fp32"),
        # the mixed form users pick by default, at the benchmark shape
        dict(_case("run", 40, 400, "bf16x3", count=180000, at=1.0), name="large_bf16x3"),
        # the mixed-precision benchmark's No with a smaller basis, a segment
        dict(_case("run", 60, 240, "bf16x3", count=60000), name="wide_bf16x3"),
        # per-tuple E(T) and E(cT) of a range: two passes, per-tuple output
        dict(_case("tuples", 20, 183, count=50000, with_j=True), name="tuples_ct"),
        # complex (T), a whole small calculation
        dict(_case("run", 14, 90, complex=True), name="complex"),
        # many small systems of uneven size in one call
        dict(_case("batch", 0, 0, systems=64), name="batch_64"),
        # a request loop with small and mid-size requests in one stream
        dict(_case("serve", 0, 0, systems=10), name="serve_10"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _flop_tuple(c):
    passes = (4 if c["complex"] else 1) * (2 if c["with_j"] else 1)
    return 12.0 * c["no"] ** 3 * (c["no"] + c["nv"]) * passes


def draw(rng):
    kind = rng.choice(["run", "run", "run", "mixed", "mixed", "complex",
                       "tuples", "drop_in", "batch", "serve"])
    if kind == "batch":
        return _case("batch", 0, 0, precision=rng.choice(["fp64", "fp64", "split_fp32"]),
                     systems=rng.randint(16, 64))
    if kind == "serve":
        return _case("serve", 0, 0, precision=rng.choice(["fp64", "bf16x3"]),
                     systems=rng.randint(4, 10))
    if kind == "drop_in":
        return _case("drop_in", rng.randint(4, 16), rng.randint(20, 90))
    if kind == "complex":
        no, nv = rng.randint(5, 20), rng.randint(24, 110)
        c = _case("run", no, nv, complex=True)
    elif kind == "tuples":
        c = _case("tuples", _log_int(rng, 8, 36), _log_int(rng, 60, 240),
                  with_j=rng.random() < 0.5)
    elif kind == "mixed":
        c = _case("run", _log_int(rng, 10, 60), _log_int(rng, 80, 320),
                  rng.choice(["split_fp32", "fp32", "bf16x3", "bf16x3"]))
    else:
        c = _case("run", _log_int(rng, 4, 48), _log_int(rng, 36, 360))
    # a range of the space where the whole of it takes too long: from its
    # start, in the middle or the rest of it
    c["at"] = rng.choice([0.0, rng.random(), 1.0])
    most = 1e13 if c["precision"] == "fp64" else 2e13
    most /= 2 if c["complex"] or c["kind"] == "tuples" else 1
    count = int(min(most / _flop_tuple(c), 300000)) * rng.uniform(0.4, 1.0)
    c["count"] = int(count) if count < n_tuples(c["nv"]) else 0
    return c


# ---- shapes and ranges -----------------------------------------------------


def _mix64(z):
    z = (z + 0x9E3779B97F4A7C15) & (1 << 64) - 1
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & (1 << 64) - 1
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & (1 << 64) - 1
    return z ^ (z >> 31)


def _shapes(case):
    """[(No, Nv)] of the systems of a batch or serve case: fixed by the
    number of systems, so that every seed costs the same."""
    out = []
    for s in range(case["systems"]):
        u, v = (_mix64(7919 * case["systems"] + 2 * s + k) / 2.0 ** 64 for k in (0, 1))
        if case["kind"] == "batch":  # No 4..16, Nv 20..120, uniform
            out.append((4 + int(13 * u), 20 + int(101 * v)))
        else:  # No 8..24, Nv 40..128, log-uniform
            out.append((round(8 * 3 ** u), round(40 * 3.2 ** v)))
    return out


def _range(case):
    """(first, count) of the tuple range of a case, count None for all of
    the space; `at` places it between the start (0) and the end (1)."""
    if not case["count"]:
        return 0, None
    return int((n_tuples(case["nv"]) - case["count"]) * case["at"]), case["count"]


def _seeds(case, seed):
    return [seed * 1009 + s for s in range(max(1, case["systems"]))]


# ---- the measured calls ----------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "ctx": hip.Context(0), "seeds": _seeds(case, seed)}
    ctx = state["ctx"]
    if kind == "drop_in":
        state["tensors"] = _host_tensors(case["no"], case["nv"], seed)
    elif kind == "batch":
        state["systems"] = [ctx.upload_synthetic(no, nv, s)
                            for (no, nv), s in zip(_shapes(case), state["seeds"])]
    elif kind != "serve":
        # a program that runs one mixed form keeps only its operands
        ctx.set_option("operand_store", OPERAND_STORE[case["precision"]])
        if case["complex"]:
            state["system"] = ctx.upload_synthetic_complex(
                case["no"], case["nv"], state["seeds"][0], with_j=case["with_j"])
        else:
            state["system"] = ctx.upload_synthetic(
                case["no"], case["nv"], state["seeds"][0], with_j=case["with_j"])
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind, precision = case["kind"], case["precision"]
    first, count = _range(case) if kind in ("run", "tuples") else (0, None)
    if kind == "run":
        e, e_ct = ctx.run(state["system"], precision, first=first, count=count)
        return {"e": np.float64(e), "e_ct": np.float64(e_ct)}
    if kind == "tuples":
        if count is None:
            count = n_tuples(case["nv"])
        e, e_ct = ctx.tuple_energies(state["system"], first, count, precision,
                                     with_ct=True)
        return {"e": e, "e_ct": e_ct}
    if kind == "batch":
        return {"e": ctx.batch_run(state["systems"], precision)}
    if kind == "serve":
        with serve.Server(ctx, hbm_budget_gb=50.0, precision=precision) as srv:
            ids = [srv.submit_synthetic(no, nv, s)
                   for (no, nv), s in zip(_shapes(case), state["seeds"])]
            done = srv.drain(ids)
        return {"e": np.array([done[r]["energy"] for r in ids])}
    system = ctx.upload(case["no"], case["nv"], state["tensors"])
    e, e_ct = ctx.run(system, precision)
    ctx.release(system)
    return {"e": np.float64(e), "e_ct": np.float64(e_ct)}


def work(case):
    """Bytes and operations of one pass: every input element that the range
    needs once (a range of n tuples reaches at most 6 n ordered virtual
    pairs and 3 n virtual orbitals), the doubles contractions
    (12 No^3 (No + Nv) per tuple) and the energies of the No^3 points."""
    if case["kind"] in ("batch", "serve"):
        one = [work(_case("run", no, nv, case["precision"])) for no, nv in _shapes(case)]
        return {k: sum(w[k] for w in one) for k in ("bytes", "flops")}
    no, nv = case["no"], case["nv"]
    n = case["count"] or n_tuples(nv)
    parts = 2 if case["complex"] else 1
    sets = 2 if case["with_j"] else 1
    pairs, orbitals = min(nv * nv, 6 * n), min(nv, 3 * n)
    operand = 8 if case["kind"] == "drop_in" else OPERAND_BYTES[case["precision"]]
    size = operand * parts * (sets * pairs * no * nv            # Vabci, Jabci
                              + (1 + sets) * orbitals * no ** 3  # Vijka, Jijka
                              + orbitals * nv * no * no)         # Tabij
    size += 8 * parts * (pairs * no * no + no * nv + no + nv)    # Vabij, Tai, eps
    out = 16 * n if case["kind"] == "tuples" else 16
    points = no * (no + 1) * (no + 2) / 6
    return {"bytes": float(size + out),
            "flops": n * (_flop_tuple(case) + 60.0 * points * parts * sets)}


# ---- inputs ----------------------------------------------------------------


def _host_tensors(no, nv, seed):
    """Host tensors in the library's upload layout (column-major, first index
    fastest), as flat float64 arrays."""
    r = np.random.default_rng(seed)

    def pairs(sd):
        # symmetric under (a, i) <-> (b, j): C order [j, i, b, a]
        x = r.normal(0.0, sd, (no, no, nv, nv))
        swapped = x.transpose(1, 0, 3, 2)
        key = np.arange(nv)[None, :] + nv * np.arange(no)[:, None]  # [i, a]
        own = key[None, :, None, :] <= key[:, None, :, None]
        return np.where(own, x, swapped).reshape(-1)

    return {
        "ei": r.uniform(-1.5, -0.3, no), "ea": r.uniform(0.1, 3.0, nv),
        "Tai": r.normal(0.0, 1e-3, nv * no), "Tabij": pairs(1e-2), "Vabij": pairs(5e-2),
        "Vijka": r.normal(0.0, 5e-2, no ** 3 * nv), "Vabci": r.normal(0.0, 5e-2, nv ** 3 * no),
    }


# The seeded generator of the synthetic systems, in plain torch: SplitMix64
# streams and Box-Muller normals, one stream per tensor.

_TENSOR = {"ei": 0, "ea": 1, "Tai": 2, "Tabij": 3, "Vabij": 4, "Vijka": 5,
           "Vabci": 6, "Jijka": 7, "Jabci": 8}
_SPREAD = {"Tai": 1e-3, "Tabij": 1e-2}


def _signed(z):
    return z - (1 << 64) if z >= 1 << 63 else z


def _shift(x, n):
    return (x >> n) & ((1 << (64 - n)) - 1)


def _mix(z):
    z = (z ^ _shift(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ _shift(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ _shift(z, 31)


def _stream(seed, tensor):
    # (_mix64 adds the increment before it mixes)
    z = _mix64(seed) ^ ((tensor + 1) * 0xD1B54A32D192ED03 & (1 << 64) - 1)
    return _mix64(z - 0x9E3779B97F4A7C15 & (1 << 64) - 1)


def _uniform(stream, n):
    bits = _mix((n + 1) * _signed(0x9E3779B97F4A7C15) + _signed(stream))
    return (_shift(bits, 11).double() + 0.5) * 2.0 ** -53


def _normal(stream, n):
    u, v = _uniform(stream, 2 * n), _uniform(stream, 2 * n + 1)
    return torch.sqrt(-2.0 * torch.log(u)) * torch.cos(2.0 * math.pi * v)


class _Synthetic:
    """Elements of a seeded synthetic system (its imaginary part with
    imag=True) by their column-major index."""

    def __init__(self, no, nv, seed, device, imag=False):
        self.no, self.nv, self.device, self.imag = no, nv, device, imag
        self.seed = seed

    def _index(self, axes):
        """Sum of range * stride over axes [(n, stride), ...], one tensor
        dimension each."""
        out = torch.zeros((), dtype=torch.int64, device=self.device)
        for d, (n, stride) in enumerate(axes):
            shape = [1] * len(axes)
            shape[d] = n
            out = out + torch.arange(n, device=self.device).reshape(shape) * stride
        return out

    def get(self, name, axes):
        if name in ("ei", "ea"):
            if self.imag:
                return torch.zeros([n for n, _ in axes], dtype=torch.float64, device=self.device)
            stream = _stream(self.seed, _TENSOR[name])
            scale, shift = (1.2, -1.5) if name == "ei" else (2.9, 0.1)
            return scale * _uniform(stream, self._index(axes)) + shift
        stream = _stream(self.seed, _TENSOR[name] | (16 if self.imag else 0))
        rows = max(1, int(4e7 / math.prod(n for n, _ in axes[1:])))
        out = torch.empty([n for n, _ in axes], dtype=torch.float64, device=self.device)
        for r in range(0, axes[0][0], rows):
            n = min(rows, axes[0][0] - r)
            at = self._index([(n, axes[0][1])] + list(axes[1:])) + r * axes[0][1]
            if name in ("Tabij", "Vabij"):
                at = self._mirror(at)
            out[r:r + n] = _SPREAD.get(name, 5e-2) * _normal(stream, at)
        return out

    def _mirror(self, at):
        no, nv = self.no, self.nv
        a, b = at % nv, at // nv % nv
        i, j = at // (nv * nv) % no, at // (nv * nv * no)
        other = b + nv * a + nv * nv * j + nv * nv * no * i
        return torch.where(a + nv * i > b + nv * j, other, at)


class _Given:
    """The same access to host tensors."""

    def __init__(self, no, nv, tensors, device):
        self.t = {k: torch.from_numpy(np.asarray(v)).to(device) for k, v in tensors.items()}

    def get(self, name, axes):
        return torch.as_strided(self.t[name], [n for n, _ in axes],
                                [s for _, s in axes]).contiguous()


# ---- the energies in 64 bits -----------------------------------------------


class _Energies:
    """Per-tuple (T) energies of one system from the closed-shell formulas,

      W = P [ sum_E T[a,E,i,j] V[b,c,E,k] - sum_L H[i,j,L,b] T[a,c,L,k] ]
      Z = W + t[a,i] V[b,c,j,k] + t[b,j] V[a,c,i,k] + t[c,k] V[a,b,i,j]
      E = 2 f sum_ijk W (4 Z + Z_jki + Z_kij - 2 (Z_ikj + Z_jik + Z_kji)) / D

    P the sum over the six simultaneous permutations of (a,i), (b,j), (c,k);
    D = eps_a + eps_b + eps_c - eps_i - eps_j - eps_k; f one half where two
    virtual indices agree.  Complex systems take conj(H) in W, conj(W) in E
    and the real part."""

    def __init__(self, no, nv, parts, with_j):
        self.no, self.nv, self.with_j = no, nv, with_j
        n2 = nv * nv

        def tensor(name, axes):
            x = [p.get(name, axes) for p in parts]
            return torch.complex(*x) if len(x) == 2 else x[0]

        def integrals(v, h):
            hole = tensor(h, [(nv, no ** 3), (no, no * no), (no, no), (no, 1)])
            return (tensor(v, [(nv, 1), (nv, nv), (nv, n2), (no, n2 * nv)]),
                    hole.conj().resolve_conj())

        # T, V2 [a, b, i, j]; V [b, c, E, k]; H [x, L, j, i]
        axes = [(nv, 1), (nv, nv), (no, n2), (no, n2 * no)]
        self.T, self.V2 = tensor("Tabij", axes), tensor("Vabij", axes)
        self.sets = [integrals("Vabci", "Vijka")]
        if with_j:
            self.sets.append(integrals("Jabci", "Jijka"))
        self.t = tensor("Tai", [(nv, 1), (no, nv)])
        self.ei, self.ea = tensor("ei", [(no, 1)]), tensor("ea", [(nv, 1)])

    def _w(self, integrals, a, b, c):
        """W[b, c, i, j, k] of the tuples (a, b, c) for slices b and c."""
        V, H = integrals
        T, no = self.T, self.no
        nb, nc = b.stop - b.start, c.stop - c.start

        def mul(x, y, dims, order):
            """x [rows.., K] times y [K, columns..]: the product's axes (sizes
            dims) permuted to b, c, i, j, k."""
            z = x.reshape(-1, x.shape[-1]) @ y.reshape(y.shape[0], -1)
            return z.reshape(dims).permute(order)

        Ta, Tb, Tc = T[a], T[b], T[c]  # [E, i, j], [b, E, j, i], ...
        w = mul(Ta.permute(1, 2, 0), V[b, c].permute(2, 0, 1, 3),
                (no, no, nb, nc, no), (2, 3, 0, 1, 4))                   # T[a,E,i,j] V[b,c,E,k]
        w = w + mul(Tb.permute(0, 2, 3, 1), V[a, c].permute(1, 0, 2),
                    (nb, no, no, nc, no), (0, 3, 2, 1, 4))               # T[b,E,j,i] V[a,c,E,k]
        w += mul(Ta.permute(1, 2, 0), V[c, b].permute(2, 0, 1, 3),
                 (no, no, nc, nb, no), (3, 2, 0, 4, 1))                  # T[a,E,i,k] V[c,b,E,j]
        w += mul(Tc.permute(0, 2, 3, 1), V[a, b].permute(1, 0, 2),
                 (nc, no, no, nb, no), (3, 0, 2, 4, 1))                  # T[c,E,k,i] V[a,b,E,j]
        w += mul(Tb.permute(0, 2, 3, 1), V[c, a].permute(1, 0, 2),
                 (nb, no, no, nc, no), (0, 3, 4, 1, 2))                  # T[b,E,j,k] V[c,a,E,i]
        w += mul(Tc.permute(0, 2, 3, 1), V[b, a].permute(1, 0, 2),
                 (nc, no, no, nb, no), (3, 0, 4, 2, 1))                  # T[c,E,k,j] V[b,a,E,i]
        # hole terms: H[x] is [L, q, p] for H[p,q,L,x], T[x, y] is [L, n]
        rows = lambda h: h.permute(*range(h.dim() - 3), -1, -2, -3)  # noqa: E731  [.., p, q, L]
        Ha, Hb, Hc = rows(H[a]), rows(H[b]), rows(H[c])
        w -= mul(Hb, Ta[c].permute(1, 0, 2), (nb, no, no, nc, no), (0, 3, 1, 2, 4))
        w -= mul(Ha, T[b, c].permute(2, 0, 1, 3), (no, no, nb, nc, no), (2, 3, 1, 0, 4))
        w -= mul(Hc, Ta[b].permute(1, 0, 2), (nc, no, no, nb, no), (3, 0, 1, 4, 2))
        w -= mul(Ha, T[c, b].permute(2, 0, 1, 3), (no, no, nc, nb, no), (3, 2, 1, 4, 0))
        w -= mul(Hc, T[b, a].permute(1, 0, 2), (nc, no, no, nb, no), (3, 0, 4, 1, 2))
        w -= mul(Hb, T[c, a].permute(1, 0, 2), (nb, no, no, nc, no), (0, 3, 4, 2, 1))
        return w

    def block(self, a, b, c):
        """[E, E(cT)] of the tuples (a, b, c) as [b, c] matrices."""
        t, V2, ei, ea = self.t, self.V2, self.ei, self.ea
        ws = [self._w(s, a, b, c) for s in self.sets]
        z = ws[0] + t[a][:, None, None] * V2[b, c][:, :, None]
        z += t[b][:, None, None, :, None] * V2[a, c][None, :, :, None, :]
        z += t[c][None, :, None, None, :] * V2[a, b][:, None, :, :, None]
        d = (ea[a] + ea[b][:, None] + ea[c][None])[:, :, None, None, None] - (
            ei[:, None, None] + ei[None, :, None] + ei)
        p = lambda i, j, k: z.permute(0, 1, 2 + i, 2 + j, 2 + k)  # noqa: E731
        # axes of z in the order that reads z at the permuted point
        y = 4.0 * z + p(2, 0, 1) + p(1, 2, 0) - 2.0 * (p(0, 2, 1) + p(1, 0, 2) + p(2, 1, 0))
        y /= d
        nv = torch.arange(self.nv, device=z.device)
        half = 1.0 - 0.5 * ((nv[b] == a)[:, None] | (nv[b][:, None] == nv[c][None])).double()
        return [2.0 * half * (w.conj() * y).real.sum((2, 3, 4)) if w.is_complex()
                else 2.0 * half * (w * y).sum((2, 3, 4)) for w in ws]

    def over(self, first, count):
        """Per-tuple energies [set][tuple] of the range, in index order."""
        no, nv = self.no, self.nv
        last = first + count
        out = [torch.zeros(count, dtype=torch.float64, device=self.T.device) for _ in self.sets]
        most = max(1, int(6e7 / no ** 3 / (2 if self.T.is_complex() else 1)))
        start = 0  # index of the first tuple of a
        for a in range(nv):
            rows = [nv - b - (b == a) for b in range(a, nv)]  # tuples of (a, b)
            begin = start + np.concatenate([[0], np.cumsum(rows)])
            start = int(begin[-1])
            hit = [b for b in range(a, nv)
                   if begin[b - a] < last and begin[b - a + 1] > first and rows[b - a]]
            while hit:
                b = slice(hit[0], min(hit[-1] + 1, hit[0] + max(1, most // (nv - hit[0]))))
                c = slice(b.start, nv)
                if hit[0] == hit[-1]:  # one row: only its part of the range
                    skip = b.start + (b.start == a)
                    lo = max(0, first - int(begin[b.start - a])) + skip
                    c = slice(lo, min(nv, last - int(begin[b.start - a]) + skip))
                e = self.block(a, b, c)
                for x in range(b.start, b.stop):
                    lo = max(c.start, x + (x == a))
                    at = int(begin[x - a]) + lo - x - (x == a)
                    n = c.stop - lo
                    skip, stop = max(0, first - at), min(n, last - at)
                    if stop > skip:
                        for k, ek in enumerate(e):
                            row = ek[x - b.start, lo - c.start + skip:lo - c.start + stop]
                            out[k][at + skip - first:at + stop - first] = row
                hit = [x for x in hit if x >= b.stop]
        return out


def _exact_system(case, no, nv, seed, tensors=None):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if tensors is not None:
        parts = [_Given(no, nv, tensors, device)]
    else:
        parts = [_Synthetic(no, nv, seed, device, imag)
                 for imag in ((False, True) if case["complex"] else (False,))]
    first, count = _range(case) if case["kind"] in ("run", "tuples") else (0, None)
    got = _Energies(no, nv, parts, case["with_j"]).over(
        first, n_tuples(nv) if count is None else count)
    return [got[0], got[-1]]


def exact(case, seed):
    if work(case)["flops"] > (2e14 if torch.cuda.is_available() else 2e11):
        return None  # would take too long
    kind = case["kind"]
    if kind in ("batch", "serve"):
        return {"e": np.array([-_exact_system(case, no, nv, s)[0].sum().item()
                               for (no, nv), s in zip(_shapes(case), _seeds(case, seed))])}
    tensors = _host_tensors(case["no"], case["nv"], seed) if kind == "drop_in" else None
    e, e_ct = _exact_system(case, case["no"], case["nv"], _seeds(case, seed)[0], tensors)
    if kind == "tuples":
        return {"e": e.cpu().numpy(), "e_ct": e_ct.cpu().numpy()}
    return {"e": np.float64(-e.sum().item()), "e_ct": np.float64(-e_ct.sum().item())}
