"""Workloads of the hopping-term library that are timed and compared: what a
lattice program has it do, through the package's public entry points, on
device-resident fields (or on host arrays where the entry takes them).

A case is a dict of plain values: `kind` names the entry, the rest its sizes
and options.  `listed()` holds the fixed ones, `draw(rng)` another of the same
ranges, `prepare(case, seed)` the objects a program holds before the call,
`run(state)` one pass, `work(case)` the bytes and operations the pass cannot
do without, and `exact(case, seed)` its outputs as plain torch computes them
in 64 bits.

Fields come back as torch tensors over the library's own device memory, in the
stored type and order [slot][16-byte chunk][minor index][reals of the chunk]
(minor index = right-hand side * Ls + s), so that a pass copies nothing.
"""
import ctypes
import os
import random

import numpy as np
import torch

import gridbench_amd as gbx

DTYPE = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
NBYTES = {"f64": 8, "f32": 4, "f16": 2, "bf16": 2}
TUNED = os.path.join(os.path.dirname(gbx.LIB_PATH), "tuned_mi355x.jsonl")
KAPPA = 0.12          # the hopping parameter of bench.py's solves
TOL = 1e-10
SHAPES = (8, 12, 16)  # extents and Ls of the uneven batch


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # The benchmark's headline: 24^4 x Ls16 FP64, one right-hand side, on
        # the traversal order, spin basis and cached launch shape it uses.
        dict(name="dhop_f64_24", kind="dhop", prec="f64", dims="24x24x24x24", Ls=16, nrhs=1, dag=False, comp12=False,
             tuned=True),
        # The smallest call: the reference's CPU configuration, where launch
        # and call overhead count.
        dict(name="dhop_f64_8", kind="dhop", prec="f64", dims="8x8x8x8", Ls=8, nrhs=1, dag=False, comp12=False,
             tuned=False),
        # An ordinary ragged lattice that nobody tuned, daggered, FP32.
        dict(name="dhop_f32_ragged", kind="dhop", prec="f32", dims="20x18x10x14", Ls=10, nrhs=1, dag=True, comp12=False,
             tuned=False),
        # Multi-right-hand-side applications of a measurement program.
        dict(name="dhop_bf16_16rhs", kind="dhop", prec="bf16", dims="16x16x16x24", Ls=12, nrhs=16, dag=False,
             comp12=False, tuned=False),
        dict(name="dhop_f32_8rhs", kind="dhop", prec="f32", dims="16x16x16x16", Ls=16, nrhs=8, dag=False, comp12=False,
             tuned=False),
        # One half of the even-odd operator, x - kappa^2 DhopEO: what a
        # red-black solver applies.
        dict(name="eo_xpay_f64", kind="eo", prec="f64", dims="24x24x24x24", Ls=12, nrhs=1, dag=False),
        # The domain-wall operator and the inverse of its fifth-dimension term.
        dict(name="dwf_apply_f64", kind="dwf", prec="f64", dims="24x24x24x24", Ls=16, nrhs=1, dag=False),
        dict(name="dwf_mooee_inv_f32", kind="mooee", prec="f32", dims="24x24x24x24", Ls=16, nrhs=1, dag=True),
        # Whole solves to 1e-10 with low-precision inner iterations.
        dict(name="cg_f16", kind="cg", inner="f16", dims="16x16x16x24", Ls=8),
        dict(name="dwf_solve_f32", kind="dwf_solve", inner="f32", dims="16x16x16x16", Ls=12),
        # Many uneven lattices in one call.
        dict(name="batch_f32", kind="batch", prec="f32", n=12, shapes=505),
        # The reference's own entry, on host arrays in its layout (the
        # benchmark's program calls it once with many repetitions).
        dict(name="dslash_host_f64", kind="host", prec="f64", dims="16x16x16x16", Ls=8, nsimd=4, rrii=False, nrep=10),
    ]


def _extent(rng, lo, hi, step=1):
    """An extent spread over the logarithm of lo .. hi, a multiple of step."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    return max(lo, v - v % step)


def _dims(rng, lo, hi, step=1):
    return "x".join(str(_extent(rng, lo, hi, step)) for _ in range(4))


def draw(rng):
    kind = rng.choice(["dhop", "dhop", "dhop", "dhop", "eo", "dwf", "mooee", "cg", "dwf_solve", "batch", "host"])
    dag = rng.random() < 0.5
    if kind == "dhop":
        prec = rng.choice(["f64", "f32", "f16", "bf16"])
        nrhs = rng.choice([1, 1, 1, 2, 3, 4, 6, 8, 12, 16])
        return dict(kind=kind, prec=prec, dims=_dims(rng, 4, 22 if nrhs == 1 else 14), Ls=_extent(rng, 4, 20), nrhs=nrhs,
                    dag=dag, comp12=rng.random() < 0.25, tuned=False)
    if kind == "eo":
        return dict(kind=kind, prec=rng.choice(["f64", "f32"]), dims=_dims(rng, 4, 24, 2), Ls=_extent(rng, 4, 20), nrhs=1,
                    dag=dag)
    if kind in ("dwf", "mooee"):
        return dict(kind=kind, prec=rng.choice(["f64", "f32"]), dims=_dims(rng, 4, 22), Ls=_extent(rng, 4, 24),
                    nrhs=rng.choice([1, 1, 2]), dag=dag)
    if kind in ("cg", "dwf_solve"):
        return dict(kind=kind, inner=rng.choice(["f32", "f16", "bf16"]), dims=_dims(rng, 6, 16, 2), Ls=_extent(rng, 4, 12))
    if kind == "batch":
        return dict(kind=kind, prec=rng.choice(["f32", "f16", "bf16"]), n=rng.randint(3, 12), shapes=rng.randrange(1 << 20))
    return dict(kind=kind, prec=rng.choice(["f64", "f32"]), dims=_dims(rng, 4, 16, 4), Ls=_extent(rng, 4, 16),
                nsimd=rng.choice([1, 2, 4]), rrii=rng.random() < 0.3, nrep=rng.choice([1, 4, 10]))


def _parse(dims):
    return tuple(int(v) for v in dims.split("x"))


def _batch_shapes(case):
    r = random.Random(case["shapes"])
    return [((r.choice(SHAPES),) * 4, r.choice(SHAPES), r.randint(1, 4)) for _ in range(case["n"])]


# ------------------------------------------------------------------ the inputs
def _rng(seed, stream):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + stream)


def _spinor(dims, Ls, seed, stream, prec):
    """One right-hand side, N(0,1) values of the storage type as float64: [V][Ls][4][3][2], x fastest."""
    V = int(np.prod(dims))
    x = torch.randn((V, Ls, 4, 3, 2), generator=_rng(seed, stream), device="cuda", dtype=torch.float32)
    return x.to(DTYPE[prec]).double()


def _links(dims, seed, prec="f64"):
    """Doubled random SU(3) field as complex128 [V][8][3][3], its values of the storage type."""
    V = int(np.prod(dims))
    z = torch.randn((V, 4, 2, 3, 2), generator=_rng(seed, 0), device="cuda", dtype=torch.float64)
    z = torch.view_as_complex(z)
    a = z[:, :, 0] / z[:, :, 0].abs().square().sum(-1, keepdim=True).sqrt()
    b = z[:, :, 1] - (a.conj() * z[:, :, 1]).sum(-1, keepdim=True) * a
    b = b / b.abs().square().sum(-1, keepdim=True).sqrt()
    u = torch.stack([a, b, torch.linalg.cross(a, b).conj()], 2)  # [V][4][3][3]
    grid = u.reshape(dims[::-1] + (4, 3, 3))
    back = [torch.roll(grid[..., mu, :, :], 1, 3 - mu).mH for mu in range(4)]
    d = torch.stack([grid[..., mu, :, :] for mu in range(4)] + back, 4).reshape(V, 8, 3, 3)
    return torch.view_as_complex(torch.view_as_real(d).contiguous().to(DTYPE[prec]).double())


def _host(x):
    x = torch.view_as_real(x) if x.is_complex() else x
    return x.contiguous().cpu().numpy()


def _half(dims, x, parity):
    """The sites of one parity of [V, ...], in the checkerboarded order of a red-black half."""
    c = [torch.arange(n, device=x.device) for n in dims[::-1]]
    p = sum(torch.meshgrid(*c, indexing="ij")).reshape(-1) % 2
    return x[p == parity]


# -------------------------------------------------------- fields as torch views
class _Memory:
    def __init__(self, field, address, shape, typestr):
        self.field = field  # the tensor's storage holds this object, and so the field
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(address, False), version=2)


TYPESTR = {"f64": "<f8", "f32": "<f4", "f16": "<f2", "bf16": "<i2"}


def _view(field):
    """The field's device memory as a tensor [slot][chunk][minor][real].  The
    handle is a pointer to the library's field object, whose device address
    follows the geometry pointer and four 32-bit shape words."""
    prec = gbx.PREC_NAMES[field.prec]
    address = ctypes.c_uint64.from_address(field.h.value + 24).value
    per = 16 // NBYTES[prec]
    shape = (field.geom.volume, 24 // per, field.Ls * field.nrhs, per)
    assert int(np.prod(shape)) * NBYTES[prec] == field.nbytes
    t = torch.as_tensor(_Memory(field, address, shape, TYPESTR[prec]), device="cuda")
    assert t.data_ptr() == address
    t = t.view(torch.bfloat16) if prec == "bf16" else t
    t.field = field
    return t


def _upload(field, lex):
    """lex: one [V][Ls][4][3][2] tensor per right-hand side."""
    for r, x in enumerate(lex):
        field.upload_rhs(r, _host(x))
    return field


def _sites(geom):
    """The lexicographic site of every slot, as uploads place them."""
    f = gbx.SpinorField(geom, 1, 1, "f64")
    V = geom.volume
    f.upload(np.repeat(np.arange(V, dtype=np.float64), 24))
    site = _view(f)[:, 0, 0, 0].long()
    torch.cuda.synchronize()  # before the field goes
    return site


def _stored(lex, geom, prec):
    """Right-hand sides [V][Ls][4][3] complex128 laid out as the field stores them, in 64 bits."""
    slot = _sites(geom)
    per = 16 // NBYTES[prec]
    out = []
    for x in lex:
        x = torch.view_as_real(x)[slot]  # [slot][Ls][4][3][2]
        out.append(x.reshape(x.shape[0], x.shape[1], 24 // per, per).transpose(1, 2))
    return torch.cat(out, 2)


# --------------------------------------------------------------------- prepare
class State:
    pass


def _geometry(case, dims):
    # the block order the benchmark uses for FP64 single-right-hand-side rows
    return gbx.Geometry(dims, block=(4, 6, 6, 12)) if case.get("tuned") else gbx.Geometry(dims)


def prepare(case, seed):
    s = State()
    s.case = case
    kind = case["kind"]
    if kind == "batch":
        s.U, s.src, s.dst = [], [], []
        for i, (dims, Ls, nrhs) in enumerate(_batch_shapes(case)):
            g = gbx.Geometry(dims)
            p = case["prec"]
            s.U.append(gbx.GaugeField(g, p).upload(_host(_links(dims, seed * 64 + i, p))))
            s.src.append(_upload(gbx.SpinorField(g, Ls, nrhs, p),
                                 [_spinor(dims, Ls, seed * 64 + i, 1 + r, p) for r in range(nrhs)]))
            s.dst.append(gbx.SpinorField(g, Ls, nrhs, p))
        s.batch = gbx.Batch(s.U, s.dst, s.src)
        s.out = [_view(f) for f in s.dst]
        return s
    dims, Ls = _parse(case["dims"]), case["Ls"]
    if kind == "host":
        dt = np.float64 if case["prec"] == "f64" else np.float32
        U, x = _links(dims, seed, case["prec"]), _spinor(dims, Ls, seed, 1, case["prec"])
        V = int(np.prod(dims))
        s.U = _lanes(case, dims, torch.view_as_real(U).reshape(V, 1, 72, 2)).cpu().numpy().astype(dt)
        s.src = _lanes(case, dims, x.reshape(V, Ls, 12, 2)).cpu().numpy().astype(dt)
        s.dst = np.zeros_like(s.src)
        s.nbr, s.prm = gbx.table_generate(dims, case["nsimd"], Ls)
        s.nsite = V // case["nsimd"]
        return s
    if kind == "mooee":
        s.geom = gbx.Geometry(dims)
        s.src, s.dst = (gbx.SpinorField(s.geom, Ls, case["nrhs"], case["prec"]) for _ in range(2))
        _upload(s.src, [_spinor(dims, Ls, seed, 1 + r, case["prec"]) for r in range(case["nrhs"])])
        s.out = _view(s.dst)
        return s
    if kind in ("eo", "dwf_solve"):
        pair = gbx.Geometry.rb_pair(dims)
        prec = case.get("prec", "f64")
        U = _host(_links(dims, seed, prec))
        x = _spinor(dims, Ls, seed, 1, prec)
        halves = [_half(dims, x, p) for p in (0, 1)]
        s.pair = pair
        if kind == "eo":  # out_e = x_e - kappa^2 DhopEO psi_o
            s.U = gbx.GaugeField(pair[0], prec).upload(U)
            s.x, s.dst = (gbx.SpinorField(pair[0], Ls, 1, prec) for _ in range(2))
            s.src = _upload(gbx.SpinorField(pair[1], Ls, 1, prec), [halves[1]])
            _upload(s.x, [halves[0]])
            s.out = _view(s.dst)
            return s
        s.U = [gbx.GaugeField(g, "f64").upload(U) for g in pair]
        s.lo = [gbx.GaugeField(g, case["inner"]).upload(U) for g in pair]
        s.b = [_upload(gbx.SpinorField(g, Ls, 1, "f64"), [h]) for g, h in zip(pair, halves)]
        s.x = [gbx.SpinorField(g, Ls, 1, "f64") for g in pair]
        s.out = [_view(f) for f in s.x]
        return s
    s.geom = _geometry(case, dims)
    if kind == "cg":
        U = _host(_links(dims, seed))
        s.U, s.lo = (gbx.GaugeField(s.geom, p).upload(U) for p in ("f64", case["inner"]))
        s.b = _upload(gbx.SpinorField(s.geom, Ls, 1, "f64"), [_spinor(dims, Ls, seed, 1, "f64")])
        s.x = gbx.SpinorField(s.geom, Ls, 1, "f64")
        s.out = _view(s.x)
        return s
    prec, nrhs = case["prec"], case["nrhs"]
    s.U = gbx.GaugeField(s.geom, prec, case.get("comp12", False)).upload(_host(_links(dims, seed, prec)))
    s.src, s.dst = (gbx.SpinorField(s.geom, Ls, nrhs, prec) for _ in range(2))
    _upload(s.src, [_spinor(dims, Ls, seed, 1 + r, prec) for r in range(nrhs)])
    if case.get("tuned"):
        s.src.set_basis(gbx.BASIS_TDIAG)
        gbx.tune(s.U, s.dst, s.src, cache_path=TUNED)
    s.out = _view(s.dst)
    return s


# ------------------------------------------------------------------------- run
def run(s):
    c = s.case
    kind = c["kind"]
    if kind == "dhop":
        gbx.dhop(s.U, s.dst, s.src, dag=c["dag"])
    elif kind == "eo":
        gbx.dhop_xpay(s.U, s.dst, s.x, s.src, 1.0, -KAPPA * KAPPA, dag=c["dag"])
    elif kind == "dwf":
        gbx.dwf_apply(s.U, s.dst, s.src, dag=c["dag"])
    elif kind == "mooee":
        gbx.dwf_mooee(s.dst, s.src, inv=True, dag=c["dag"])
    elif kind == "cg":
        s.x.zero()
        gbx.cg_solve(s.U, s.lo, s.x, s.b, KAPPA, tol=TOL)
    elif kind == "dwf_solve":
        for f in s.x:
            f.zero()
        gbx.dwf_solve_eo(s.U, s.lo, s.x, s.b, tol=TOL)
    elif kind == "batch":
        s.batch.run()
    else:
        gbx.dslash_kernel(c["nrep"], s.U, s.dst, s.src, s.nbr, s.nsite, c["Ls"], s.prm, c["nsimd"], rrii=c["rrii"])
        return s.dst
    return s.out


# ------------------------------------------------------------------------ work
def _dhop_work(V, Ls, nrhs, b, reals=18, extra=0):
    """Spinor in and out (and `extra` more fields) and the links once; 1320 flop a point."""
    n = V * Ls * nrhs
    return (48 + 24 * extra) * b * n + 8 * reals * b * V, 1320 * n


def work(case):
    kind = case["kind"]
    if kind == "batch":
        w = [_dhop_work(int(np.prod(d)), Ls, r, NBYTES[case["prec"]]) for d, Ls, r in _batch_shapes(case)]
        return {"bytes": sum(v[0] for v in w), "flops": sum(v[1] for v in w)}
    V, Ls = int(np.prod(_parse(case["dims"]))), case["Ls"]
    b = NBYTES[case.get("prec", "f64")]
    if kind == "dhop":
        n, f = _dhop_work(V, Ls, case["nrhs"], b, 12 if case["comp12"] else 18)
    elif kind == "eo":
        n, f = _dhop_work(V // 2, Ls, 1, b, extra=1)
        f += 48 * V // 2 * Ls
    elif kind == "dwf":
        n, f = _dhop_work(V, Ls, case["nrhs"], b)
        f += 96 * V * Ls * case["nrhs"]
    elif kind == "mooee":
        n, f = 48 * b * V * Ls * case["nrhs"], 96 * V * Ls * case["nrhs"]
    elif kind == "host":
        # host arrays across the bus once, then nrep applications
        n, f = _dhop_work(V, Ls, 1, b)
        n, f = n * (1 + case["nrep"]), f * case["nrep"]
    else:
        # About 60 (Wilson) and 65 (domain-wall) inner iterations reach the
        # tolerance; each is two operator applications in the inner precision
        # and reads and writes the CG vectors (x, r, p) once.
        it, lo = (60 if kind == "cg" else 65), NBYTES[case["inner"]]
        n, f = _dhop_work(V, Ls, 1, lo)
        vec = 24 * V * Ls * 6 * 4
        if kind == "dwf_solve":
            vec //= 2
        n, f = it * (2 * n + vec), it * 2 * f
    return {"bytes": n, "flops": f}


# ----------------------------------------------------------------------- exact
# gamma_mu in the chiral basis: row a holds one entry, in column COL[mu][a].
COL = ((3, 2, 1, 0), (3, 2, 1, 0), (2, 3, 0, 1), (2, 3, 0, 1))
VAL = ((1j, 1j, -1j, -1j), (-1, 1, 1, -1), (1j, -1j, -1j, 1j), (1, 1, 1, 1))


def _hop(U, dims, x, dag=False):
    """Dhop of one right-hand side: U [V][8][3][3], x [V][Ls][4][3], complex128."""
    V, Ls = x.shape[:2]
    out = torch.zeros_like(x)
    for d in range(8):
        mu, ax = d & 3, 3 - (d & 3)
        y = torch.roll(x.reshape(dims[::-1] + (Ls, 4, 3)), -1 if d < 4 else 1, ax).reshape(x.shape)
        h = torch.stack([sum(U[:, d, i, j, None, None] * y[..., j] for j in range(3)) for i in range(3)], -1)
        sign = (-1 if d < 4 else 1) * (-1 if dag else 1)
        out += h
        for a in range(4):
            out[:, :, a] += (sign * VAL[mu][a]) * h[:, :, COL[mu][a]]
    return out


def _mooee_matrices(Ls, dag):
    """The fifth-dimension term on the upper and the lower two spins, [Ls][Ls]."""
    m = torch.zeros((2, Ls, Ls), dtype=torch.float64)
    for s in range(Ls):
        m[:, s, s] = 5.0 - gbx.DWF_M5
        m[0, s, (s - 1) % Ls] += gbx.DWF_MASS if s == 0 else -1.0
        m[1, s, (s + 1) % Ls] += gbx.DWF_MASS if s == Ls - 1 else -1.0
    return (m.mT if dag else m).cuda()


def _fifth(m, x):
    """Apply [2][Ls][Ls] to the s index of [V][Ls][4][3]."""
    out = torch.zeros_like(x)
    for s in range(x.shape[1]):
        for t in range(x.shape[1]):
            for h in (0, 1):
                if m[h, s, t] != 0:
                    out[:, s, 2 * h:2 * h + 2] += m[h, s, t] * x[:, t, 2 * h:2 * h + 2]
    return out


def _conjugate_gradient(normal, b):
    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), r.abs().square().sum()
    stop = 1e-30 * float(rr)
    for _ in range(3000):
        if float(rr) <= stop:
            break
        q = normal(p)
        a = rr / (p.conj() * q).sum().real
        x += a * p
        r -= a * q
        new = r.abs().square().sum()
        p = r + (new / rr) * p
        rr = new
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        out = []
        for i, (dims, Ls, nrhs) in enumerate(_batch_shapes(case)):
            U = _links(dims, seed * 64 + i, case["prec"])
            x = [torch.view_as_complex(_spinor(dims, Ls, seed * 64 + i, 1 + r, case["prec"])) for r in range(nrhs)]
            out.append(_stored([_hop(U, dims, v) for v in x], gbx.Geometry(dims), case["prec"]))
        return out
    dims, Ls = _parse(case["dims"]), case["Ls"]
    prec = case.get("prec", "f64")
    x = [torch.view_as_complex(_spinor(dims, Ls, seed, 1 + r, prec)) for r in range(case.get("nrhs", 1))]
    if kind == "mooee":
        m = torch.linalg.inv(_mooee_matrices(Ls, case["dag"]).cpu()).cuda()
        return _stored([_fifth(m, v) for v in x], gbx.Geometry(dims), prec)
    U = _links(dims, seed, prec)
    if kind == "host":
        y = torch.view_as_real(_hop(U, dims, x[0])).reshape(-1, Ls, 12, 2)
        return _lanes(case, dims, y).cpu().numpy()
    if kind == "dhop":
        if case["comp12"]:
            U = torch.cat([U[:, :, :2], torch.linalg.cross(U[:, :, 0], U[:, :, 1]).conj()[:, :, None]], 2)
        y = [_hop(U, dims, v, case["dag"]) for v in x]
        if case["tuned"]:  # the stored spin basis: sums and differences of the upper and lower spins
            y = [torch.cat([v[:, :, :2] + v[:, :, 2:], v[:, :, :2] - v[:, :, 2:]], 2) * 0.5 ** 0.5 for v in y]
        return _stored(y, _geometry(case, dims), prec)
    if kind == "eo":
        pair = gbx.Geometry.rb_pair(dims)
        y = x[0] - KAPPA * KAPPA * _hop(U, dims, x[0], case["dag"])
        return _stored([_half(dims, y, 0)], pair[0], prec)
    if kind == "dwf":
        m = _mooee_matrices(Ls, case["dag"])
        return _stored([_fifth(m, v) - 0.5 * _hop(U, dims, v, case["dag"]) for v in x], gbx.Geometry(dims), prec)
    if kind == "cg":
        y = _conjugate_gradient(lambda v: _wilson(U, dims, _wilson(U, dims, v, False), True), x[0])
        return _stored([y], gbx.Geometry(dims), prec)
    m, md = _mooee_matrices(Ls, False), _mooee_matrices(Ls, True)
    y = _conjugate_gradient(lambda v: _domain_wall(U, dims, md, _domain_wall(U, dims, m, v, False), True),
                            _domain_wall(U, dims, md, x[0], True))
    pair = gbx.Geometry.rb_pair(dims)
    return [_stored([_half(dims, y, p)], pair[p], prec) for p in (0, 1)]


def _wilson(U, dims, v, dag):
    return v - KAPPA * _hop(U, dims, v, dag)


def _domain_wall(U, dims, m, v, dag):
    return torch.einsum("hst,vthac->vshac", m.to(v.dtype), v.reshape(v.shape[0], v.shape[1], 2, 2, 3)).reshape(
        v.shape) - 0.5 * _hop(U, dims, v, dag)


def _lanes(case, dims, x):
    """[V][Ls][n complex][2] in the reference's vector layout: nsimd lanes a
    vector, split by twos over T, Z, ..., and the real and imaginary parts of
    a lane side by side, or all real parts first."""
    n, simd = case["nsimd"], [1, 1, 1, 1]
    d = 3
    while n > 1:
        simd[d] *= 2
        n //= 2
        d = (d + 3) % 4
    shape = []
    for d in (3, 2, 1, 0):
        shape += [simd[d], dims[d] // simd[d]]
    y = x.reshape(tuple(shape) + x.shape[1:])  # lane and outer coordinates of T, Z, Y, X, then [Ls][n][2]
    order = (1, 3, 5, 7, 8, 9) + ((10, 0, 2, 4, 6) if case["rrii"] else (0, 2, 4, 6, 10))
    return y.permute(order).reshape(-1)
