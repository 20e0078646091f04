"""The work that a user of the prover has it do, at the sizes that its configurations name and over the ranges around them.

A case is a dict with a "kind" and that kind's sizes:

  fr_mul   elementwise product of two full-width field tensors
  fc       a fully connected layer: the matrix product and zkFC::prove of it
  commit   Pedersen row commitments of an integer weight matrix, as points with z = 1
  open     a commitment opened at a point (Commitment::open): every point of the proof
  lookup   range-table lookup: multiplicities and the lookup argument
  mapping  lookup in a table of function values: outputs, multiplicities, argument
  rescale  division by a power of two with its remainder range proof
  attn     attention with its proof: Q K^T, softmax by table segments, times V
  layer    a whole decoder layer computed and proved, weight openings included

Everything goes through the C entry points of the class layer (libzkllm_prover.so) on tensors that are on the GPU; field elements come
back as int32 limbs, eight to an element, points as 36.  All results are exact.
"""
import ctypes
import importlib

import numpy as np
import torch

pkg = importlib.import_module("zkllm-ccs2024_amd")

_P, _U, _I = ctypes.c_void_p, ctypes.c_uint32, ctypes.c_int
_lib = None


def _prover():
    global _lib
    if _lib is None:
        lib = pkg.load_prover()
        for name in ("zkp_fr_from_i32", "zkp_fr_from_fr", "zkp_fr_devptr", "zkp_fr_binop", "zkp_fr_matmul", "zkp_commitment_random", "zkp_commit_int",
                     "zkp_g1_binop", "zkp_g1_devptr", "zkp_rescale_prove", "zkp_attn", "zkp_layer_create", "zkp_layer_create_random", "zkp_layer_run"):
            getattr(lib, name).restype = _P
        for name in ("zkp_fr_size", "zkp_g1_size"):
            getattr(lib, name).restype = _U
        for name in ("zkp_transcript_size", "zkp_transcript_g1_size"):
            getattr(lib, name).restype = ctypes.c_long
        _ok(lib.zkp_init(_I(0)), lib)
        _lib = lib
    return _lib


def _ok(rc, lib=None):
    if rc != 0:
        raise RuntimeError("prover error: " + (lib or _lib).zkp_last_error().decode())


def _ptr(a):
    return _P(a.ctypes.data)


class _Handle:
    """A tensor of field elements ("fr"), of points ("g1") or a layer that lives until nothing refers to it any more."""
    LIMBS = {"fr": 8, "g1": 36}

    def __init__(self, h, what="fr"):
        if not h:
            raise RuntimeError("prover error: " + _lib.zkp_last_error().decode())
        self.h, self.what = _P(h), what

    def __del__(self):
        getattr(_lib, "zkp_%s_free" % self.what)(self.h)

    @property
    def __cuda_array_interface__(self):
        n = getattr(_lib, "zkp_%s_size" % self.what)(self.h)
        return {"shape": (n, self.LIMBS[self.what]), "typestr": "<i4", "data": (getattr(_lib, "zkp_%s_devptr" % self.what)(self.h), False), "version": 2}

    def tensor(self):
        """The tensor's limbs where they are, as int32; the memory stays this handle's."""
        return torch.as_tensor(self, device="cuda")


def _from_ints(t):
    a = t.to(torch.int32).cpu().numpy()
    return _Handle(_prover().zkp_fr_from_i32(_ptr(a), _U(a.size)))


def _elements(rs, n):
    """n field elements drawn as a challenge stream draws them: uniform limbs below the modulus' top limb."""
    a = rs.randint(0, 1 << 32, (n, 8), dtype=np.uint64).astype(np.uint32)
    a[:, 7] %= 1944954707
    return a


def _field_tensor(gen, n):
    t = torch.randint(-(1 << 31), 1 << 31, (n, 8), generator=gen, device="cuda", dtype=torch.int64)
    t[:, 7] = t[:, 7].remainder(1944954707)
    a = t.to(torch.int32).cpu().numpy()
    return _Handle(_prover().zkp_fr_from_fr(_ptr(a), _U(n)))


def _normal(gen, n, std, limit=None):
    t = torch.empty(n, device="cuda").normal_(0.0, 1.0, generator=gen).mul_(std).round_()
    return t.clamp_(-limit, limit) if limit else t


def _weights(gen, n):
    """fixed-point weights: N(0, 0.02) at scale 2^16"""
    return _from_ints(_normal(gen, n, 0.02 * 65536))


def _record(lib, seed):
    lib.zkp_seed(_U(seed))
    lib.zkp_transcript_begin()


def _transcript(lib):
    out = np.empty((lib.zkp_transcript_size(), 8), np.int32)
    lib.zkp_transcript_get(_ptr(out))
    lib.zkp_transcript_end()
    return out


def _log2(n):
    return (n - 1).bit_length()


def listed():
    return [
        # one of the headline figures: field products over a 2048 x 4096 tensor
        {"name": "fr_mul_2048x4096", "kind": "fr_mul", "n": 2048 * 4096},
        # the smallest layer anybody proves (and the smoke test's): all launches and waits
        {"name": "fc_16x64x64", "kind": "fc", "batch": 16, "inputs": 64, "outputs": 64},
        # a mid-sized layer with no dimension a power of two
        {"name": "fc_300x1000x2750", "kind": "fc", "batch": 300, "inputs": 1000, "outputs": 2750},
        # a 7B-shape projection at 2048 tokens
        {"name": "fc_2048x4096x4096", "kind": "fc", "batch": 2048, "inputs": 4096, "outputs": 4096},
        # the commitment of a 7B-shape weight, the headline's points per second
        {"name": "commit_11008x4096", "kind": "commit", "rows": 11008, "generators": 4096},
        # the opening of a 4096 x 4096 weight under out_features << 5 generators
        {"name": "open_128x131072", "kind": "open", "rows": 128, "generators": 1 << 17},
        # lookup of 2^22 queries in a table of 2^16
        {"name": "lookup_2e22_2e16", "kind": "lookup", "queries": 1 << 22, "table": 1 << 16},
        # an activation table over a ragged hidden tensor
        {"name": "mapping_300x2750", "kind": "mapping", "queries": 300 * 2750, "table": 1 << 18},
        # the rescaling behind a ragged matrix product
        {"name": "rescale_300x1000", "kind": "rescale", "n": 300 * 1000, "log_factor": 16},
        # one head at 2048 tokens
        {"name": "attn_1x2048x128", "kind": "attn", "heads": 1, "seq": 2048, "dim": 128},
        # a layer of the test configuration: hundreds of short launches and their host work
        {"name": "layer_small", "kind": "layer", "model": "small", "seq": 16, "embed": 32, "heads": 2, "hidden": 64},
        # the headline's decoder layer at 2048 tokens, with half its width: three such layers fit the card beside each other
        {"name": "layer_2048x2048", "kind": "layer", "model": "random", "seq": 2048, "embed": 2048, "heads": 16, "hidden": 5504},
    ]


def _spread(rng, low, high):
    """a whole number, its logarithm uniform between those of low and high"""
    return max(low, min(high, int(round(low * (high / low) ** rng.random()))))


def draw(rng):
    kind = rng.choice(("fr_mul", "fc", "commit", "open", "lookup", "mapping", "rescale", "attn", "layer"))
    if kind == "fr_mul":
        return {"kind": kind, "n": _spread(rng, 1 << 10, 1 << 25)}
    if kind == "fc":
        return {"kind": kind, "batch": _spread(rng, 1, 2048), "inputs": _spread(rng, 64, 4096), "outputs": _spread(rng, 64, 11008)}
    if kind == "commit":
        return {"kind": kind, "rows": _spread(rng, 1, 11008), "generators": 1 << rng.randint(6, 12)}
    if kind == "open":
        lg = rng.randint(6, 17)
        return {"kind": kind, "rows": 1 << rng.randint(0, min(7, 24 - lg)), "generators": 1 << lg}
    if kind == "lookup":
        lq = rng.randint(9, 24)
        return {"kind": kind, "queries": 1 << lq, "table": _spread(rng, 1 << 6, 1 << min(16, lq))}
    if kind == "mapping":
        n = _spread(rng, 1 << 10, 1 << 24)
        return {"kind": kind, "queries": n, "table": 1 << rng.randint(8, min(20, _log2(n)))}
    if kind == "rescale":
        n = _spread(rng, 1 << 9, 1 << 24)
        return {"kind": kind, "n": n, "log_factor": rng.randint(6, min(20, _log2(n)))}
    if kind == "attn":
        while True:
            c = {"kind": kind, "heads": 1 << rng.randint(0, 5), "seq": 1 << rng.randint(6, 11), "dim": 1 << rng.randint(5, 7)}
            if 1 << 15 <= c["heads"] * c["seq"] ** 2 <= 1 << 25:
                return c
    if rng.random() < 0.5:
        heads = 1 << rng.randint(1, 2)
        return {"kind": kind, "model": "small", "seq": 1 << rng.randint(4, 6), "embed": heads << rng.randint(4, 5), "heads": heads, "hidden": _spread(rng, 64, 256)}
    log_seq = rng.randint(9, 10)
    log_embed = rng.randint(20 - log_seq, 11)
    return {"kind": kind, "model": "random", "seq": 1 << log_seq, "embed": 1 << log_embed, "heads": 1 << (log_embed - rng.randint(6, 7)),
            "hidden": _spread(rng, 2 << log_embed, 3 << log_embed)}


def _layer_config(case):
    """the arguments of zkp_layer_create*: the scales of the drivers for the "random" model, those of the tests' layer for the small one"""
    seq, embed, heads, hidden = (case[k] for k in ("seq", "embed", "heads", "hidden"))
    if case["model"] == "small":
        cu = [seq, embed, heads, hidden, 1 << 8, 1 << 10, 1 << 7, 1, 0, 1024, 1, 3, 1 << 8, 1 << 8, 1 << 8, 0]
        cf = [1 << 16, -512, 64.0, 16.0, 1e-5, 256.0, 1 << 6, 1 << 8]
    else:
        table = min(1 << 22, 1 << _log2(seq * hidden))
        cu = [seq, embed, heads, hidden, 1 << 16, 1 << 20, 1 << 20, 1, 0, table, 1, 3, 1 << 8, 1 << 20, 1 << 20, heads]
        cf = [1 << 32, -(table >> 1), 4096.0, 16.0, 1e-5, 65536.0, 1 << 18, 1 << 22]
    return np.array(cu, np.uint32), np.array(cf, np.float64)


def prepare(case, seed):
    lib = _prover()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rs = np.random.RandomState(seed % (1 << 31))
    kind, s = case["kind"], {"case": case, "seed": seed % (1 << 31)}
    if kind == "fr_mul":
        s["a"], s["b"] = _field_tensor(gen, case["n"]), _field_tensor(gen, case["n"])
    elif kind == "fc":      # activations of unit variance at scale 2^16
        s["X"] = _from_ints(_normal(gen, case["batch"] * case["inputs"], 65536.0, 1 << 20))
        s["W"] = _weights(gen, case["inputs"] * case["outputs"])
    elif kind in ("commit", "open"):
        lib.zkp_seed(_U(s["seed"]))
        s["gens"] = _Handle(lib.zkp_commitment_random(_U(case["generators"])), "g1")
        s["t"] = _weights(gen, case["rows"] * case["generators"])
        if kind == "open":
            s["com"] = _Handle(lib.zkp_commit_int(s["gens"].h, s["t"].h), "g1")
            s["u"] = _elements(rs, _log2(case["rows"]) + _log2(case["generators"]))
    elif kind == "lookup":
        n = case["table"]
        s["S"] = _from_ints(torch.randint(0, n, (case["queries"],), generator=gen, device="cuda") - n // 2)
        s["one"], s["two"] = _elements(rs, 2), _elements(rs, 2 * _log2(case["queries"]))
    elif kind == "mapping":      # queries around the middle of the table, values as an activation's
        n, low = case["table"], -(case["table"] // 2)
        s["S"] = _from_ints(_normal(gen, case["queries"], n / 16.0, n // 2 - 1))
        x = torch.arange(low, low + n, device="cuda", dtype=torch.float64) * (16.0 / n)
        s["values"] = _from_ints((torch.nn.functional.silu(x) * 65536).round())
        s["one"], s["two"] = _elements(rs, 3), _elements(rs, 2 * _log2(case["queries"]))
    elif kind == "rescale":
        s["X"] = _from_ints(_normal(gen, case["n"], 2.0 ** 27, (1 << 31) - 128))
    elif kind == "attn":
        n = case["heads"] * case["seq"] ** 2
        s["digit"] = 1 << min(20, _log2(n))
        s["scale"] = 1 << min(32, 2 * _log2(s["digit"]) - 4)      # of the scores: the table segments have to hold them
        std = s["scale"] ** 0.5
        s["Q"], s["K"], s["V"] = (_from_ints(_normal(gen, case["heads"] * case["seq"] * case["dim"], std)) for _ in range(3))
    else:
        cu, cf = _layer_config(case)
        lib.zkp_seed(_U(s["seed"]))
        E, H = case["embed"], case["hidden"]
        if case["model"] == "small":
            w_std = 0.25 * (32.0 / E) ** 0.5      # scores and gates keep to the tables' ranges at every width
            w = [np.full(E, 256, np.int32) if shape == (1, E) else np.round(rs.normal(0, w_std, shape) * 256).astype(np.int32)
                 for shape in ((1, E), (E, E), (E, E), (E, E), (E, E), (1, E), (E, H), (E, H), (H, E))]
            s["layer"] = _Handle(lib.zkp_layer_create(_ptr(cu), _ptr(cf), *[_ptr(x) for x in w], _U(5)), "layer")
            std = 256.0
        else:
            s["layer"] = _Handle(lib.zkp_layer_create_random(_ptr(cu), _ptr(cf), _U(s["seed"]), _U(5)), "layer")
            std = 65536.0
        s["X"] = _from_ints(_normal(gen, case["seq"] * E, std))
    return s


def run(s):
    lib, case = _lib, s["case"]
    kind = case["kind"]
    if kind == "fr_mul":
        return _Handle(lib.zkp_fr_binop(_I(2), s["a"].h, s["b"].h)).tensor()
    if kind == "fc":
        dims = _U(case["inputs"]), _U(case["outputs"])
        y = _Handle(lib.zkp_fr_matmul(s["X"].h, s["W"].h, _U(case["batch"]), *dims))
        claim = np.zeros(8, np.int32)
        _record(lib, s["seed"])
        _ok(lib.zkp_zkfc_prove(s["X"].h, s["W"].h, y.h, *dims, _ptr(claim)))
        return {"Y": y.tensor(), "proof": _transcript(lib), "claim_W": claim}
    if kind == "commit":
        com = _Handle(lib.zkp_commit_int(s["gens"].h, s["t"].h), "g1")
        return _Handle(lib.zkp_g1_binop(_I(3), com.h, com.h), "g1").tensor()
    if kind == "open":
        k = s["u"].shape[0]
        points, count, value = np.zeros((3 * k + 1, 36), np.int32), _I(0), np.zeros(8, np.int32)
        _ok(lib.zkp_open(s["gens"].h, s["t"].h, s["com"].h, _ptr(s["u"]), _I(k), _ptr(points), ctypes.byref(count), _ptr(value)))
        return {"points": points[:count.value], "value": value}
    if kind == "lookup":
        k, last = s["two"].shape[0] // 2, np.zeros(8, np.int32)
        _record(lib, s["seed"])
        _ok(lib.zkp_range_prove(s["S"].h, _I(-(case["table"] // 2)), _U(case["table"]), _ptr(s["one"][0]), _ptr(s["one"][1]), _ptr(s["two"][:k]), _ptr(s["two"][k:]), _ptr(last)))
        return {"proof": _transcript(lib), "claim": last}
    if kind == "mapping":
        k, last = s["two"].shape[0] // 2, np.zeros(8, np.int32)
        y, m = _P(), _P()
        _record(lib, s["seed"])
        _ok(lib.zkp_mapping(s["S"].h, _I(-(case["table"] // 2)), _U(case["table"]), s["values"].h, *[_ptr(x) for x in s["one"]], _ptr(s["two"][:k]), _ptr(s["two"][k:]),
                            ctypes.byref(y), ctypes.byref(m), _ptr(last)))
        return {"outputs": _Handle(y.value).tensor(), "multiplicities": _Handle(m.value).tensor(), "proof": _transcript(lib), "claim": last}
    if kind == "rescale":
        _record(lib, s["seed"])
        out = _Handle(lib.zkp_rescale_prove(s["X"].h, _U(1 << case["log_factor"])))
        return {"out": out.tensor(), "proof": _transcript(lib)}
    if kind == "attn":
        bs, thetas = np.array([1 << 8, s["digit"], s["digit"]], np.uint32), np.array([1 << 18, 1 << 22], np.float64)
        last = np.zeros(8, np.int32)
        _record(lib, s["seed"])
        out = _Handle(lib.zkp_attn(s["Q"].h, s["K"].h, s["V"].h, _U(case["heads"]), _U(case["seq"]), _U(case["seq"]), _U(case["dim"]), _I(0 if case["heads"] == 1 else 2),
                                   _ptr(bs), _I(3), _U(1), _U(0), ctypes.c_uint64(s["scale"]), ctypes.c_uint64(1), _ptr(thetas), _I(2), _ptr(last)))
        return {"out": out.tensor(), "proof": _transcript(lib), "claim": last}
    _record(lib, s["seed"])
    out = _Handle(lib.zkp_layer_run(s["layer"].h, s["X"].h, None))
    points = np.empty((lib.zkp_transcript_g1_size(), 36), np.int32)
    if points.size:
        lib.zkp_transcript_g1_get(_ptr(points))
    return {"out": out.tensor(), "points": points, "proof": _transcript(lib)}


def work(case):
    """Bytes: 32 an element read or written, 144 a point.  Operations: two for each 32-bit limb product (136 in a field product modulo r, 300
    modulo p; 64 a term of a field dot product kept unreduced) and two for each int8 product where small integers are multiplied."""
    fr, fp, kind = 2 * 136, 2 * 300, case["kind"]
    if kind == "fr_mul":
        return {"bytes": 96 * case["n"], "flops": fr * case["n"]}
    if kind == "fc":
        b, i, o = case["batch"], case["inputs"], case["outputs"]
        # three digits of an activation times two of a weight; each tensor folded once
        return {"bytes": 32 * (b * i + i * o + b * o), "flops": 2 * 6 * b * i * o + 2 * 64 * (b * i + i * o + b * o)}
    if kind in ("commit", "open"):
        r, g = case["rows"], case["generators"]
        if kind == "commit":      # two 8-bit windows of a 14-bit weight, a mixed addition of 11 products each
            return {"bytes": 32 * r * g + 144 * (g + r), "flops": 2 * 11 * fp * r * g}
        # the scalars' rows folded; a generator pair folded with a 255-bit scalar: 128 doublings and 64 additions with the endomorphism
        return {"bytes": 32 * r * g + 144 * g, "flops": 2 * 64 * r * g + g * fp * (128 * 7 + 64 * 11)}
    if kind == "lookup":      # about ten products a query over all the rounds
        return {"bytes": 32 * (case["queries"] + case["table"]), "flops": 10 * fr * case["queries"]}
    if kind == "mapping":
        return {"bytes": 32 * (2 * case["queries"] + 2 * case["table"]), "flops": 10 * fr * case["queries"]}
    if kind == "rescale":
        return {"bytes": 64 * case["n"], "flops": 12 * fr * case["n"]}
    if kind == "attn":
        h, m, d = case["heads"], case["seq"], case["dim"]
        return {"bytes": 32 * 4 * h * m * d, "flops": 2 * 9 * 2 * h * m * m * d + 35 * fr * h * m * m}
    b, e, h, f = case["seq"], case["embed"], case["heads"], case["hidden"]
    macs = 4 * b * e * e + 3 * b * e * f
    queries = 3 * h * b * b + 9 * b * e + 4 * b * f
    gens = (5 * e << 5) + 2 * (1 << _log2(f << 5))
    return {"bytes": 32 * (4 * e * e + 3 * e * f + 2 * b * e) + 144 * gens, "flops": 2 * 6 * macs + 2 * 9 * 2 * b * b * e + 10 * fr * queries + gens * fp * (128 * 7 + 64 * 11)}


def tolerance(case):
    return "exact"
