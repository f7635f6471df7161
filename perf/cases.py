"""The work that a user of this library has it do, as cases that can be timed.

A case is a contraction or a permutation through the public API (`hiptensor_amd.api`).  What a
program keeps is made in `prepare` (handle, plan, workspace, device tensors, the scalars); `run`
is the one call that such a program repeats.

A contraction is written like an einsum whose tensors list their modes in memory order, fastest
first: "abxy,ijxy->abij" is a packed column-major product of rank-2 groups,
"yxba,yxji->jiba" the same one in the row-major layout that a descriptor without strides has.
`pad` is the padding of the leading dimension of C and D, in elements.
A permutation B[modes permuted] = alpha * A is packed, first mode fastest (what the API assumes);
mode k of B is mode perm[k] of A.
"""
import math

import torch

from hiptensor_amd import api
from hiptensor_amd import workloads as wl

TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "f64": torch.float64,
         "c32": torch.complex64, "c64": torch.complex128}
COMPUTE = {"f16": api.HIPTENSOR_COMPUTE_32F, "bf16": api.HIPTENSOR_COMPUTE_32F, "f32": api.HIPTENSOR_COMPUTE_32F,
           "f64": api.HIPTENSOR_COMPUTE_64F, "c32": api.HIPTENSOR_COMPUTE_C32F, "c64": api.HIPTENSOR_COMPUTE_C64F}


def contraction(name, dtype, modes, extents, bilinear, pad=0):
    alpha, beta = (1.0 + 0.5j, 0.25 - 0.75j) if dtype in ("c32", "c64") else (1.5, -0.5)
    case = {"kind": "contract", "dtype": dtype, "modes": modes, "extents": extents, "bilinear": bilinear, "pad": pad,
            "alpha_re": alpha.real, "alpha_im": alpha.imag, "beta_re": beta.real, "beta_im": beta.imag}
    return dict(case, name=name) if name else case


def permutation(name, dtype, lens, perm, alpha):
    case = {"kind": "permute", "dtype": dtype, "lens": "x".join(map(str, lens)), "perm": "".join(map(str, perm)), "alpha": alpha}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest calls: a network of small tensors contracted pair by pair, or a step of an iterative solver on
        # small matrices, where launch and host time are all there is
        contraction("f32_256", "f32", "abxy,ijxy->abij", "a16 b16 i16 j16 x16 y16", True),
        # an ordinary size that is nobody's multiple of anything, in the default (row-major) layout of a descriptor
        # without strides: a contraction between two activations or two correlation tensors
        contraction("bf16_rowmajor_ragged", "bf16", "yxba,yxji->jiba", "a25 b39 i15 j101 x21 y37", True),
        # the large dense product of deep-learning work, f16 in the packed column-major layout ...
        contraction("f16_4096", "f16", "abxy,ijxy->abij", "a64 b64 i64 j64 x64 y64", False),
        # ... and bf16 with an accumulated output in the row-major one
        contraction("bf16_rowmajor_4096", "bf16", "yxba,yxji->jiba", "a64 b64 i64 j64 x64 y64", True),
        # quantum chemistry: doubles-amplitude update in double precision
        contraction("f64_1920x1920x768", "f64", "abxy,ijxy->abij", "a48 b40 i48 j40 x32 y24", True),
        # circuit simulation and signal processing: complex single precision
        contraction("c32_1024x1024x512", "c32", "abxy,ijxy->abij", "a32 b32 i32 j32 x32 y16", True),
        # a tensor-network contraction whose tensors come out of earlier steps in whatever order those left
        # them, into a padded output; the largest product here
        contraction("f16_rank6_permuted", "f16", "yaxcbz,kxizyj->abcijk", "a32 b7 c24 i24 j9 k32 x17 y8 z30", True, pad=8),
        # free and contracted modes interleaved, odd extents
        contraction("f16_interleaved", "f16", "axby,ixjy->abij", "a15 b323 i15 j323 x7 y143", False),
        # few columns against a large operand (a decode step, a projection onto a few vectors): read once
        contraction("f16_skinny_n16", "f16", "abxy,ixy->abi", "a128 b64 i16 x128 y64", False),
        # a small result of a long reduction (a Gram matrix, the gradient of a weight over many samples)
        contraction("f32_long_k", "f32", "abxy,ijxy->abij", "a16 b16 i16 j16 x256 y256", False),
        # change of storage order of a large tensor between two steps
        permutation("perm_f32_1GiB", "f32", (512, 64, 128, 64), (2, 0, 3, 1), 1.5),
        # ... and of a small one with odd extents
        permutation("perm_f32_sample", "f32", (33, 32, 34, 35), (2, 3, 1, 0), 1.0),
    ]


# -- drawn cases ---------------------------------------------------------------------------------

FLOP_RATE = {"f16": 2.5e15, "bf16": 2.5e15, "f32": 157e12, "c32": 157e12, "f64": 78e12, "c64": 78e12}  # nominal, dense
NOMINAL_S = 110e-6  # a drawn case's time at the nominal rates is below this: the largest listed ones stand at 120 us (contraction) ...
PERM_ELEMS = (1 << 14, 1 << 28)  # ... and at 1 GiB (permutation)


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _split(rng, n, modes):
    """Extents of `modes` modes whose product is about n."""
    w = [rng.uniform(0.4, 1.0) for _ in range(modes)]
    return [max(1 if n < 2 ** modes else 2, int(round(n ** (x / sum(w))))) for x in w]


def _shuffled(rng, s):
    s = list(s)
    rng.shuffle(s)
    return "".join(s)


def _interleaved(a, b):
    out = "".join(x + y for x, y in zip(a, b))
    return out + a[len(b):] + b[len(a):]


def _draw_contraction(rng):
    while True:
        dtype = rng.choice(["f16", "f16", "f16", "bf16", "bf16", "bf16", "f32", "f32", "f32", "f64", "f64", "c32", "c32", "c64"])
        shape = rng.choice(["small", "ordinary", "ordinary", "large", "large", "skinny", "long"])
        if shape == "small":
            m, n, k = (_between(rng, 8, 300) for _ in range(3))
        elif shape == "ordinary":
            m, n, k = (_between(rng, 128, 2048) for _ in range(3))
        elif shape == "large":
            m, n, k = (_between(rng, 800, 6000) for _ in range(3))
        elif shape == "skinny":
            m, n, k = _between(rng, 1024, 16384), _between(rng, 1, 64), _between(rng, 512, 8192)
            if rng.random() < 0.5:
                m, n = n, m
        else:
            m, n, k = _between(rng, 32, 512), _between(rng, 32, 512), _between(rng, 8192, 131072)
        groups, ext = [], {}
        for letters, size in (("abc", m), ("ijk", n), ("xyz", k)):
            r = min(3, max(1, int(math.log2(max(2, size)))))
            g = letters[: rng.randint(1, r)]
            ext.update(zip(g, _split(rng, size, len(g))))
            groups.append(g)
        if rng.random() < 0.5 and shape != "small":  # extents that suit a machine: each a multiple of 4
            ext = {x: e if e < 4 else (e + 2) // 4 * 4 for x, e in ext.items()}
        gm, gn, gk = groups
        layout = rng.choice(["columns", "columns", "rows", "rows", "mixed", "permuted", "interleaved"])
        pad = 0
        if layout == "columns":
            a, b, d = gm + gk, gn + gk, gm + gn
        elif layout == "rows":
            a, b, d = (gm + gk)[::-1], (gn + gk)[::-1], (gm + gn)[::-1]
        elif layout == "mixed":
            a, b, d = rng.choice([(gm + gk, gk + gn, gm + gn), (gk + gm, gn + gk, gm + gn)])
        elif layout == "permuted":
            a, b, d, pad = _shuffled(rng, gm + gk), _shuffled(rng, gn + gk), gm + gn, rng.choice([0, 8])
        else:
            a, b, d = _interleaved(gm, gk), _interleaved(gn, gk), rng.choice([gm + gn, _interleaved(gm, gn)])
        case = contraction("", dtype, f"{a},{b}->{d}", " ".join(f"{x}{ext[x]}" for x in gm + gn + gk), rng.random() < 0.5, pad)
        w = work(case)
        if max(w["flops"] / FLOP_RATE[dtype], w["bytes"] / 8e12) <= NOMINAL_S:
            return case


def draw(rng):
    if rng.random() < 0.8:
        return _draw_contraction(rng)
    while True:
        rank = rng.randint(2, 6)
        n = _between(rng, *PERM_ELEMS)
        lens, perm = _split(rng, n, rank), list(range(rank))
        rng.shuffle(perm)
        if perm != sorted(perm) and math.prod(lens) <= PERM_ELEMS[1]:
            return permutation("", rng.choice(["f16", "f32"]), lens, perm, rng.choice([1.0, 1.5]))


# -- what a case is --------------------------------------------------------------------------------

def _contract_shape(case):
    """(modes of A, B, D as label lists in memory order, extent by label)"""
    ext = {ord(t[0]): int(t[1:]) for t in case["extents"].split()}
    ab, d = case["modes"].split("->")
    a, b = ab.split(",")
    return [ord(x) for x in a], [ord(x) for x in b], [ord(x) for x in d], ext


def _perm_shape(case):
    return [int(x) for x in case["lens"].split("x")], [int(x) for x in case["perm"]]


def work(case):
    e = wl.ELEM_BYTES[case["dtype"]]
    if case["kind"] == "permute":
        n = math.prod(_perm_shape(case)[0])
        return {"bytes": 2 * e * n, "flops": n}
    a, b, d, ext = _contract_shape(case)
    na, nb, nd = (math.prod(ext[m] for m in t) for t in (a, b, d))
    k = math.prod(ext[m] for m in a if m in b)
    return {"bytes": e * (na + nb + nd * (2 if case["bilinear"] else 1)),
            "flops": (8.0 if case["dtype"] in ("c32", "c64") else 2.0) * nd * k}


def tolerance(case):
    """A permutation multiplies each element once: exact.  A contraction: about four times the distance (2-norm) from a
    product in 64 bits that was measured over these ranges: the rounding of the result for the 16-bit types (2.1e-4 f16,
    1.7e-3 bf16, at any K), the sums' own for the others (f32 1.6e-7 at K = 256, 8e-7 at K = 65536; c32 5e-7; f64 2e-15)."""
    if case["kind"] == "permute":
        return "exact"
    return {"rel": {"f16": 8e-4, "bf16": 6.6e-3, "f32": 5e-6, "c32": 5e-6, "f64": 1e-14, "c64": 1e-14}[case["dtype"]]}


# -- running one -----------------------------------------------------------------------------------

_handle = None


def handle():
    """The library handle of this process, made at its first use."""
    global _handle
    if _handle is None:
        torch.zeros(1, device="cuda")
        _handle = api.check(api.hiptensorCreate(), "hiptensorCreate")
    return _handle


def _uniform(n, dtype, gen):
    """n values of i.i.d. uniform [-1, 1) (both parts of complex ones) on the device."""
    t = TORCH[dtype]
    real = {torch.complex64: torch.float32, torch.complex128: torch.float64}.get(t)
    if real is not None:
        return torch.view_as_complex(torch.empty(n, 2, dtype=real, device="cuda").uniform_(-1, 1, generator=gen))
    return torch.empty(n, dtype=t, device="cuda").uniform_(-1, 1, generator=gen)


def _prepare_permutation(case, gen):
    lens, perm = _perm_shape(case)
    n, t = math.prod(lens), wl.HIP_TYPE[case["dtype"]]
    h = handle()
    state = {
        "kind": "permute", "A": _uniform(n, case["dtype"], gen), "B": torch.zeros(n, dtype=TORCH[case["dtype"]], device="cuda"),
        "dA": api.check(api.hiptensorInitTensorDescriptor(h, lens, None, t), "A"),
        "dB": api.check(api.hiptensorInitTensorDescriptor(h, [lens[p] for p in perm], None, t), "B"),
        "modesA": list(range(len(lens))), "modesB": perm, "type": t,
        "alpha": wl.permutation_alpha({"scalar": case["dtype"], "alpha": case["alpha"]}),
    }
    return dict(state, a=state["A"].data_ptr(), b=state["B"].data_ptr(), stream=torch.cuda.current_stream().cuda_stream)


def _prepare_contraction(case, gen):
    a, b, d, ext = _contract_shape(case)
    dtype, compute, bil = case["dtype"], COMPUTE[case["dtype"]], case["bilinear"]
    h, t = handle(), wl.HIP_TYPE[dtype]
    lens = {"A": [ext[m] for m in a], "B": [ext[m] for m in b], "D": [ext[m] for m in d]}
    sA, sB = wl.packed_strides(lens["A"]), wl.packed_strides(lens["B"])
    sD = wl.storage_order_strides(d, ext, d, pad_after_first=case["pad"])
    dA, dB, dD = (api.check(api.hiptensorInitTensorDescriptor(h, n, s, t), "tensor")
                  for n, s in ((lens["A"], sA), (lens["B"], sB), (lens["D"], sD)))
    align = 16
    desc = api.check(api.hiptensorInitContractionDescriptor(
        h, dA, a, align, dB, b, align, dD if bil else None, d if bil else None, align if bil else 0, dD, d, align, compute), "contraction")
    find = api.check(api.hiptensorInitContractionFind(h, api.HIPTENSOR_ALGO_DEFAULT), "find")
    size = api.check(api.hiptensorContractionGetWorkspaceSize(h, desc, find, api.HIPTENSOR_WORKSPACE_RECOMMENDED), "workspace")
    plan = api.check(api.hiptensorInitContractionPlan(h, desc, find, size), "plan")
    for kind, obj in (("find", find), ("contraction", desc), ("tensor", dA), ("tensor", dB), ("tensor", dD)):
        api.destroy(kind, obj)
    span = wl.span_elems(lens["D"], sD)
    A, B = _uniform(math.prod(lens["A"]), dtype, gen), _uniform(math.prod(lens["B"]), dtype, gen)
    C = _uniform(span, dtype, gen) if bil else None
    D = torch.zeros(span, dtype=TORCH[dtype], device="cuda")  # (the padding stays zero)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda") if size else None
    alpha, beta = complex(case["alpha_re"], case["alpha_im"]), complex(case["beta_re"], case["beta_im"])
    if dtype not in ("c32", "c64"):
        alpha, beta = alpha.real, beta.real
    return {
        "kind": "contract", "handle": h, "plan": plan, "A": A, "B": B, "C": C, "D": D, "ws": ws, "ws_bytes": size,
        "alpha": wl.scalar_ctype(compute, alpha), "beta": wl.scalar_ctype(compute, beta if bil else None),
        "ptr": [x.data_ptr() if x is not None else None for x in (A, B, C, D, ws)],
        "stream": torch.cuda.current_stream().cuda_stream,
    }


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (_prepare_permutation if case["kind"] == "permute" else _prepare_contraction)(case, gen)


def run(s):
    if s["kind"] == "permute":
        api.check(api.hiptensorPermutation(handle(), s["alpha"], s["a"], s["dA"], s["modesA"], s["b"], s["dB"], s["modesB"],
                                           s["type"], s["stream"]), "hiptensorPermutation")
        return s["B"]
    A, B, C, D, ws = s["ptr"]
    api.check(api.hiptensorContraction(s["handle"], s["plan"], s["alpha"], A, B, s["beta"], C, D, ws, s["ws_bytes"], s["stream"]),
              "hiptensorContraction")
    return s["D"]
