"""The work that a user of icflow-hip has it do, as cases that can be timed and compared.

Each case is one pass over the device side of a Newton iteration (or two of them in a row)
through the C ABI or its Python mirror, on a seeded synthetic specimen:

  newton    one iteration without contact: tentative state, CZ records reset, fused assembly,
            damage counts (what icflow_amd.newton.ImplicitModel issues between two solves)
  batched   the same over many independent specimens in one call (BatchedImplicitModel)
  contact   one iteration with contact: the solver's increment, broad phase, narrow phase, tuple
            de-duplication, closest face, pattern and slots with the impacts, assembly, penalty
            response; each pass has another increment, so that the impacts change from iteration
            to iteration as they do in a Newton loop
  replay    one iteration with a fixed impact list as a captured graph (narrow phase, closest
            face, assembly, penalty response)
  fracture  the iteration after a step in which CZs failed: the CZ list and its history are
            replaced, pattern and slots are built anew; each pass has another list
  dropin    the reference host's sequence through GPUFunctionality, with its packing and host
            copies

The mesh and its grains follow from the case, the state of the nodes and the CZ history from the
seed.  Calls block, the library's default.  Every specimen has a context of its own, as the
drivers of this repository keep it.  Buffers are as large as the case can need, and outputs are
whole buffers where the state decides how much of them is used.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from icflow_amd import _lib, specimens
from icflow_amd.gpu_functionality import GPUFunctionality, stride_of

H, BETA, GAMMA = 1e-4, 0.25, 0.5        # time step of the three-point-bend beam, Newmark parameters
DIST_EPS = 1e-15
MATERIAL = _lib.SPECIMEN_PRMS


# ---- the cases ---------------------------------------------------------------------------------

def _case(name, kind, mixed, n, grains, specimens_=1):
    c = dict(kind=kind, mixed=mixed, nx=n[0], ny=n[1], nz=n[2], grains=grains, specimens=specimens_)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the small specimen of the tests, 720 tets: launches and waits are all there is
        _case("newton_small_fp64", "newton", False, (6, 5, 4), 6),
        # the three-point-bend beam, 15,360 tets: an ordinary Newton loop
        _case("newton_beam_fp64", "newton", False, (40, 8, 8), 16),
        # a larger polycrystal of odd size in mixed precision, 146,334 tets
        _case("newton_cube29_mixed", "newton", True, (29, 29, 29), 190),
        # a single large specimen, 786,786 tets, ragged in every direction
        _case("newton_large_fp64", "newton", False, (57, 43, 53), 1200),
        # a few dozen specimens side by side, FP64
        _case("batched_24_fp64", "batched", False, (12, 12, 12), 24, 24),
        # the batched workload at its full size: 256 cubes, about 3.5M tets, mixed precision
        _case("batched_256_mixed", "batched", True, (13, 13, 13), 30, 256),
        # contact on a small cube between platens (the contact study of the Newton driver)
        _case("contact_cube8_fp64", "contact", False, (8, 8, 8), 8),
        # contact on an odd block
        _case("contact_block_fp64", "contact", False, (23, 17, 19), 60),
        # compression with contact: 384,000 tets, 500 grains
        _case("contact_cube40_mixed", "contact", True, (40, 40, 40), 500),
        # the compression iteration as a captured graph, a loop that detects on a kept pair list
        _case("replay_cube40_mixed", "replay", True, (40, 40, 40), 500),
        # a beam whose CZs fail: the list of CZs shrinks, everything derived from it is rebuilt
        _case("fracture_beam_fp64", "fracture", False, (40, 8, 8), 16),
        # the reference host's own loop over this library, small specimen
        _case("dropin_beam_fp64", "dropin", False, (40, 8, 8), 16),
    ]


# cells per direction, by kind: the smallest specimens of the tests up to what a drawn case may cost
_RANGE = dict(newton=(4, 44), batched=(4, 14), contact=(4, 30), replay=(4, 34), fracture=(4, 30), dropin=(3, 14))


def draw(rng):
    kind = rng.choice(list(_RANGE))
    lo, hi = _RANGE[kind]
    edge = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    n = [max(2, round(edge * math.exp(rng.uniform(-0.4, 0.4)))) for _ in range(3)]
    while n[0] * n[1] * n[2] > hi ** 3:
        n[n.index(max(n))] -= 1
    cells = n[0] * n[1] * n[2]
    grains = max(2, round(cells / math.exp(rng.uniform(math.log(60), math.log(300)))))
    count = round(math.exp(rng.uniform(math.log(3), math.log(96)))) if kind == "batched" else 1
    return _case(None, kind, rng.random() < 0.5, n, grains, count)


# ---- specimens ---------------------------------------------------------------------------------

class _NoContact(specimens.Collection):
    """A collection whose surface is not needed: no lists of adjacent faces."""

    def _adjacency(self):
        pass


def _moved(mesh, dx):
    m = specimens.Mesh(**vars(mesh))
    m.x0 = mesh.x0 + np.array([dx, 0.0, 0.0])
    return m


@functools.lru_cache(maxsize=2)
def _specimen(kind, nx, ny, nz, grains, count):
    """The mesh of a case, cells of 2.5 mm: anchored at the bottom, or free between two platens."""
    size = (0.0025 * nx, 0.0025 * ny, 0.0025 * nz)
    if kind == "batched":
        # lognormal sizes around the case's (log-sd 0.6 in tets), 32 meshes repeated side by side
        rng = np.random.default_rng(2)
        base = []
        for _ in range(min(count, 32)):
            f = math.exp(float(np.clip(rng.normal(0.0, 0.2), -0.6, 0.4)))
            k = [max(2, round(f * v)) for v in (nx, ny, nz)]
            base.append(specimens.make_specimen(tuple(k), (0.02, 0.02, 0.02), int(rng.integers(2, 2 * grains)),
                                                int(rng.integers(1 << 30))).meshes[0])
        return _NoContact([_moved(base[k % len(base)], 0.04 * k) for k in range(count)]).finalize()
    if kind in ("contact", "replay"):
        pc = (max(1, nx * 4 // 5), max(1, ny * 4 // 5))
        return specimens.make_specimen((nx, ny, nz), size, grains, 1, platens=pc).finalize()
    col = specimens.make_specimen((nx, ny, nz), size, grains, 1)
    if kind != "dropin":
        col = _NoContact(col.meshes)
    x = col.meshes[0].x0
    col.anchored = np.isclose(x[:, 2], 0.0)
    return col.finalize()


def _mesh_of(case):
    return _specimen(case["kind"], case["nx"], case["ny"], case["nz"], case["grains"], case["specimens"])


def _state(case, col, seed):
    """Accepted state (u, v, a), increment du and CZ history of the seed."""
    consts = _lib.consts_from_prms(**MATERIAL)
    contact = case["kind"] in ("contact", "replay")
    s = specimens.synthetic_state(col, consts, seed, platen_dz=0.3 * 0.0025 if contact else 0.0)
    rng = np.random.default_rng((seed, 7))
    du = rng.normal(0.0, 0.02 * consts.deln, s.un.shape)
    du[col.anchored] = 0.0
    return consts, s, du, rng


# ---- device side -------------------------------------------------------------------------------

class _Window:
    """A run of a library buffer as a tensor; keeps the buffer's context alive."""

    def __init__(self, buf, offset, n):
        self.keep = buf
        self.__cuda_array_interface__ = dict(shape=(int(n),), typestr=buf.dtype.str, version=2,
                                             data=(buf.p.value + int(offset) * buf.dtype.itemsize, False))


def _view(buf, offset, n):
    if not n:
        return torch.empty(0, dtype=torch.float64 if buf.dtype == np.float64 else torch.int32, device="cuda")
    return torch.as_tensor(_Window(buf, offset, n), device="cuda")


class _Graph:
    def __init__(self, lib, g):
        self.lib, self.g = lib, g

    def __del__(self):
        self.lib.icf_graph_destroy(self.g)


class _Model:
    """One specimen on the device: its buffers and the calls of an iteration."""

    def __init__(self, case, seed):
        col = self.col = _mesh_of(case)
        consts, s, du, rng = _state(case, col, seed)
        gf = self.gf = GPUFunctionality(0)
        self.lib, self.ctx = gf.lib, gf.ctx
        gf.SetConstants(consts)
        gf.set_precision(_lib.ICF_MIXED if case["mixed"] else _lib.ICF_FP64)
        self.contact = case["kind"] in ("contact", "replay")
        if self.contact:
            gf.TransferStaticDataToDevice(col)
        n, ns = len(col.x0), stride_of(len(col.x0))
        self.n, self.ns, self.N = n, ns, int(col.alt.max()) + 1
        self.dn = self._soa("dn", 18, ns, [(0, col.x0)])
        acc = [(0, s.un - du), (3, s.vn), (6, s.an), (9, du)]
        self.st = self._soa("st", 12, ns, acc)
        self.alt = gf.buf("alt", n, np.int32)
        self.alt.upload(col.alt.astype(np.int32))
        self.T, self.es = len(col.elastic), stride_of(len(col.elastic))
        self.ie = self._soa("ie_el", 28, self.es, [(0, col.elastic)], np.int32)
        C = self.C = self.n_czs = len(col.czs)
        self.cs = stride_of(C)
        self.icz = self._soa("icz", 58, self.cs, [(4, col.czs)], np.int32)
        self.dcz = self._soa("dcz", 16, self.cs, [(0, s.pmax), (3, s.tmax)])
        self.rows = gf.buf("rows", self.N + 1, np.int32)
        self.rhs = gf.buf("rhs", 3 * self.N, np.float64)
        self.penalty = 1e11 * 0.0025 ** 2 * 25 / 16
        S = len(col.surf) if self.contact else 0
        self.pair_cap, self.ts = 16 * S + 4096, stride_of(S // 4 + 1024)
        self.cap = 10 * self.T + 21 * C + 1 + (6 * self.ts if self.contact else 0)
        self.nT, self.icr = 0, None
        self.cols = self._zeros("cols", self.cap, np.int32)
        self.pattern()                      # elements and CZs alone
        self.vals = self._zeros("vals", 9 * (self.nnz + (6 * self.ts if self.contact else 0)), np.float64)
        self.dmg, self.fld = ctypes.c_int(), ctypes.c_int()
        self.passes = 0
        if self.contact:
            self.pairs = self._zeros("nw_pairs", 2 * self.pair_cap, np.int32)
            self.list = self._zeros("nw_list", 2 * self.pair_cap, np.int32)
            self.nl2 = self._zeros("nw_nl2", 4 * self.ts, np.int32)
            self.impacts = self._zeros("nw_icr", 28 * self.ts, np.int32)
        if case["kind"] == "contact":       # solver increments, each with its negative
            self.dx = []
            for k in range(12):
                dx = rng.normal(0.0, 0.2 * consts.deln, 3 * self.N)
                self.dx.append([self._given("dx%d%s" % (k, "+-"[j]), v) for j, v in enumerate((dx, -dx))])
        if case["kind"] == "fracture":      # node ids and history of every CZ, twice in a row
            self.czs2 = np.concatenate([col.czs, col.czs]).T.astype(np.int32)
            self.hist2 = np.concatenate([np.concatenate([s.pmax, s.tmax], 1)] * 2).T
            self.failing = max(1, C // 50)

    def _soa(self, name, fields, stride, cols, dtype=np.float64):
        a = np.zeros(fields * stride, dtype)
        for f, v in cols:
            for k in range(v.shape[1]):
                a[(f + k) * stride:(f + k) * stride + len(v)] = v[:, k]
        b = self.gf.buf(name, a.size, dtype)
        b.upload(a)
        return b

    def _zeros(self, name, n, dtype):
        b = self.gf.buf(name, n, dtype)
        b.zero()
        return b

    def _given(self, name, a):
        b = self.gf.buf(name, a.size, a.dtype)
        b.upload(a)
        return b

    def call(self, name, *args):
        _lib.check(getattr(self.lib, name)(self.ctx, *args), self.ctx, name)

    def infer(self):
        self.call("icf_nodes_infer", self.st.p, self.ns, self.dn.p, self.ns, self.n, H, BETA, GAMMA)

    def add_dx(self):
        """The next increment: pass k adds one of twelve, or takes it back (a Gray code's changes),
        so that no two of 4,096 passes are at the same positions and none goes far."""
        self.passes = k = self.passes % 4096 + 1
        bit = (k & -k).bit_length() - 1
        sign = (k >> (bit + 1)) & 1
        if k == 4096:
            bit, sign = 11, 1               # back to the start
        self.call("icf_nodes_add_dx", self.st.p, self.ns, self.alt.p, self.n, self.dx[bit][sign].p)

    def fail_czs(self):
        """The list without another fiftieth of the CZs, and its history."""
        C = self.n_czs
        at = self.failing * (self.passes + 1) % C
        self.passes += 1
        self.C = C - self.failing
        nodes, hist = np.zeros((6, self.cs), np.int32), np.zeros((6, self.cs))
        nodes[:, :self.C] = self.czs2[:, at:at + self.C]
        hist[:, :self.C] = self.hist2[:, at:at + self.C]
        self.icz.upload(nodes.ravel(), 4 * self.cs)
        self.dcz.upload(hist.ravel())

    def pattern(self):
        nnz = ctypes.c_int()
        icr, cr = (self.icr.p, self.ts) if self.nT else (None, 0)
        self.call("icf_build_pattern", self.alt.p, self.n, self.ie.p, self.T, self.es, self.icz.p, self.C, self.cs, icr,
                  self.nT, cr, self.N, self.rows.p, self.cols.p, self.cap, ctypes.byref(nnz))
        self.call("icf_pack_pcsr", self.alt.p, self.n, self.rows.p, self.cols.p, self.N, self.ie.p, self.T, self.es,
                  self.icz.p, self.C, self.cs, icr, self.nT, cr)
        self.nnz = nnz.value

    def reset_czs(self):
        self.call("icf_pack_pcsr", self.alt.p, self.n, self.rows.p, self.cols.p, self.N, None, 0, 0, self.icz.p, self.C,
                  self.cs, None, 0, 0)

    def assemble(self, counts=True):
        d, f = (ctypes.byref(self.dmg), ctypes.byref(self.fld)) if counts else (None, None)
        self.call("icf_assemble_elems_and_czs", self.ie.p, self.T, self.es, self.dcz.p, self.icz.p, self.C, self.cs,
                  self.dn.p, self.ns, H, self.vals.p, self.nnz, self.rhs.p, self.N, d, f)

    def respond(self):
        if self.nT:
            self.call("icf_collision_response", self.icr.p, self.dn.p, H, self.vals.p, self.rhs.p, self.nT, self.ts,
                      self.ns, self.penalty, DIST_EPS)

    def detect(self):
        """Candidate pairs, narrow phase, tuples, closest faces; the impacts' nodes into icr."""
        gf, es, q, t = self.gf, self.gf.el_all_stride, ctypes.c_longlong(), ctypes.c_int()
        self.call("icf_broad_phase", self.dn.p, self.ns, gf.g_ie.p, es, len(self.col.surf), 1, self.pairs.p,
                  self.pair_cap, ctypes.byref(q))
        self.Q, self.nT, self.icr = q.value, 0, None
        if not self.Q:
            return
        self.call("icf_d2d", self.list.p, 0, self.pairs.p, 0, 8 * self.Q)
        self.call("icf_narrow_phase", self.Q, self.dn.p, gf.g_ie.p, self.list.p, es, self.ns)
        self.call("icf_nl2set", self.list.p, self.pairs.p, self.Q, gf.g_ie.p, es, self.nl2.p, self.ts,
                  ctypes.byref(t))
        if not t.value:
            return
        self.nT, self.icr = t.value, self.impacts
        self.closest()
        self.call("icf_d2d", self.icr.p, 0, self.nl2.p, 0, 16 * self.ts)

    def closest(self):
        gf = self.gf
        self.call("icf_find_closest_face", self.nT, self.ts, self.nl2.p, self.dn.p, gf.g_ie.p, gf.g_ifc.p, self.ns,
                  gf.el_all_stride, gf.fc_stride)

    def outputs(self):
        cs, ns = self.cs, self.ns
        return dict(vals=_view(self.vals, 0, self.vals.n), rhs=_view(self.rhs, 0, 3 * self.N),
                    F=_view(self.dn, 12 * ns, 3 * ns), dcz=_view(self.dcz, 6 * cs, 10 * cs),
                    flags=_view(self.icz, 0, 4 * cs), counts=[self.dmg.value, self.fld.value, self.nnz, self.nT])

    def structure(self):
        return dict(rows=_view(self.rows, 0, self.N + 1), cols=_view(self.cols, 0, self.cols.n))


def prepare(case, seed):
    if case["kind"] == "dropin":
        col = _mesh_of(case)
        consts, s, _, _ = _state(case, col, seed)
        gf = GPUFunctionality(0)
        gf.SetConstants(consts)
        gf.set_precision(_lib.ICF_MIXED if case["mixed"] else _lib.ICF_FP64)
        gf.TransferStaticDataToDevice(col)
        gf.CreateStructure(None)
        return dict(kind="dropin", gf=gf, state=s)
    m = _Model(case, seed)
    state = dict(kind=case["kind"], model=m)
    if case["kind"] == "batched":
        tet, cz, row = specimens.specimen_offsets(m.col)
        rows = m.rows.download(m.N + 1)
        offs = state["offsets"] = [np.ascontiguousarray(v, np.int32) for v in (tet, cz, row, rows[row])]
        state["worklist"] = _lib.IcfWorklist(len(tet) - 1, *[_lib.ptr(v) for v in offs])
        state["counts"] = [np.zeros(len(tet) - 1, np.int32) for _ in range(2)]
    elif case["kind"] == "replay":
        # the pair list and the impacts of a first iteration, kept; then the iteration as a graph
        m.infer()
        m.detect()
        m.pattern()
        m.kept = [m.gf.buf("kept_pairs", max(2 * m.Q, 1), np.int32), m.gf.buf("kept_tuples", 2 * m.ts, np.int32)]
        m.call("icf_d2d", m.kept[0].p, 0, m.pairs.p, 0, 8 * m.Q)
        m.call("icf_d2d", m.kept[1].p, 0, m.nl2.p, 0, 8 * m.ts)
        _replayed(m)
        m.call("icf_graph_begin")
        _replayed(m)
        g = ctypes.c_void_p()
        m.call("icf_graph_end", ctypes.byref(g))
        state["graph"] = _Graph(m.lib, g)
    return state


def _replayed(m):
    gf = m.gf
    m.infer()
    m.call("icf_d2d", m.list.p, 0, m.kept[0].p, 0, 8 * m.Q)
    m.call("icf_d2d", m.nl2.p, 0, m.kept[1].p, 0, 8 * m.ts)
    m.call("icf_narrow_phase", m.Q, m.dn.p, gf.g_ie.p, m.list.p, gf.el_all_stride, m.ns)
    if m.nT:
        m.closest()
    m.assemble(counts=False)
    m.respond()


def run(state):
    kind = state["kind"]
    if kind == "dropin":
        gf = state["gf"]
        gf.TransferNodesToGPU(state["state"])
        gf.TransferPCSR(state["state"])
        counts = gf.AssembleElemsAndCZs(H)
        vals, rhs = gf.TransferLinearSystemToHost()
        st = gf.TransferUpdatedStateToHost()
        return dict(vals=vals, rhs=rhs, F=st["F"], dcz=st["dcz"][6 * gf.cz_stride:], flags=st["icz"],
                    counts=list(counts))
    m = state["model"]
    if kind == "replay":
        m.call("icf_graph_launch", state["graph"].g)
        return dict(m.outputs(), masks=_view(m.list, 0, m.list.n), impacts=_view(m.nl2, 0, m.nl2.n))
    if kind == "contact":
        m.add_dx()
        m.infer()
        m.detect()
        m.pattern()
        m.assemble()
        m.respond()
        return dict(m.outputs(), **m.structure(), impacts=_view(m.nl2, 0, m.nl2.n))
    if kind == "fracture":
        m.fail_czs()
        m.pattern()
        m.infer()
        m.assemble()
        return dict(m.outputs(), **m.structure())
    m.infer()
    m.reset_czs()
    if kind == "newton":
        m.assemble()
        return m.outputs()
    d, f = state["counts"]
    m.call("icf_assemble_batched", ctypes.byref(state["worklist"]), m.ie.p, m.es, m.dcz.p, m.icz.p, m.cs, m.dn.p, m.ns,
           H, m.vals.p, m.rhs.p, _lib.ptr(d), _lib.ptr(f))
    return dict(m.outputs(), counts=[d.copy(), f.copy()])


# ---- what a pass cannot do without --------------------------------------------------------------

def _upper_keys(alt, units, N):
    """Distinct (row, column) pairs, row <= column, of the active nodes of each unit, as row * N + column."""
    a = alt[units]
    i, j = torch.triu_indices(a.shape[1], a.shape[1], device=a.device)
    p, q = a[:, i].reshape(-1), a[:, j].reshape(-1)
    ok = (p >= 0) & (q >= 0)
    p, q = p[ok], q[ok]
    return torch.unique(torch.minimum(p, q) * N + torch.maximum(p, q))


def _pattern(col, czs):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    alt = torch.as_tensor(col.alt, device=dev)
    N = int(alt.max()) + 1
    keys = [_upper_keys(alt, torch.as_tensor(u, device=dev), N) for u in (col.elastic, czs) if len(u)]
    return alt, N, torch.unique(torch.cat(keys))


def work(case):
    """Compulsory bytes: units' node ids and slots, CZ records, node fields, rows, blocks; pairs and
    impacts, whose number the state decides, are left out.  Operations: about 1,000 per tet
    (gradients, rotation, force, ten blocks), 1,500 per CZ (frame, law, 21 blocks), 60 per surface
    tet and direction of detection."""
    col = _mesh_of(case)
    T, C, n = len(col.elastic), len(col.czs), len(col.x0)
    _, N, keys = _pattern(col, col.czs)
    nnz = keys.numel()
    b = 96 * T + 336 * C + 144 * n + 72 * nnz + 24 * N + (12 + 15) * 8 * n
    f = 1000 * T + 1500 * C
    if case["kind"] in ("contact", "fracture"):     # pattern and slots are written too
        b += 80 * T + 168 * C + 4 * nnz + 4 * N
    if case["kind"] in ("contact", "replay"):
        b += 16 * len(col.surf)
        f += 12 * 60 * len(col.surf)
    if case["kind"] == "dropin":                    # every array crosses the bus as well
        b += 18 * 8 * n + 28 * 4 * T + (58 * 4 + 16 * 8) * C + 72 * nnz + 24 * N
    return dict(bytes=b, flops=f)


# ---- the same in plain torch, 64 bits ------------------------------------------------------------

def _material():
    """Material and PPR constants from the parameters (Park, Paulino and Roesler 2009)."""
    p = dict(_lib.MODEL_DEFAULTS, **MATERIAL)
    m = dict(p)
    a, b, ln, lt = p["alpha"], p["beta"], p["lambda_n"], p["lambda_t"]
    m["m"] = a * (a - 1) * ln ** 2 / (1 - a * ln ** 2)
    m["n"] = b * (b - 1) * lt ** 2 / (1 - b * lt ** 2)
    m["dn"] = p["phi_n"] / p["sigma_max"] * a * ln * (1 - ln) ** (a - 1) * (a / m["m"] + 1) * (a / m["m"] * ln + 1) ** (m["m"] - 1)
    m["dt"] = p["phi_t"] / p["tau_max"] * b * lt * (1 - lt) ** (b - 1) * (b / m["n"] + 1) * (b / m["n"] * lt + 1) ** (m["n"] - 1)
    if p["phi_n"] < p["phi_t"]:
        m["gn"], m["gt"] = (a / m["m"]) ** m["m"], -p["phi_t"] * (b / m["n"]) ** m["n"]
    else:
        m["gn"], m["gt"] = -p["phi_n"] * (a / m["m"]) ** m["m"], (b / m["n"]) ** m["n"]
    m["fn"], m["ft"] = max(p["phi_n"] - p["phi_t"], 0.0), max(p["phi_t"] - p["phi_n"], 0.0)
    m["lam"] = p["Y"] * p["nu"] / ((1 + p["nu"]) * (1 - 2 * p["nu"]))
    m["mu"] = p["Y"] / (2 * (1 + p["nu"]))
    return m


def _times(a, b):
    """Products of many small matrices, entry by entry."""
    return (a[..., :, :, None] * b[..., None, :, :]).sum(-2)


def _frame(a, b, c):
    """Orthonormal frame (columns) of three points."""
    d = torch.nn.functional.normalize(b - a, dim=-1)
    e = torch.nn.functional.normalize(torch.linalg.cross(b - a, c - a), dim=-1)
    return torch.stack([d, e, torch.linalg.cross(e, d)], -1)


def _law(m, opn, opt, pmax, tmax):
    """PPR tractions and tangent with unloading towards the origin and contact, per Gauss point."""
    a, b, M, N, dn, dt = m["alpha"], m["beta"], m["m"], m["n"], m["dn"], m["dt"]

    def powers(x, e, p, d):
        s = x / d
        return [(1 - s).clamp(min=0) ** (e - k) for k in range(3)], [(p / e + s) ** (p - k) for k in range(3)]

    def X(w, p, e):
        return p * w[0][0] * w[1][1] - e * w[0][1] * w[1][0]

    def Z(w, p, e):
        return (p * p - p) * w[0][0] * w[1][2] + (e * e - e) * w[0][2] * w[1][0] - 2 * e * p * w[0][1] * w[1][1]

    def n_at(x):
        return powers(x, a, M, dn)

    def t_at(x):
        return powers(x, b, N, dt)

    Tn = lambda x, y: m["gn"] / dn * X(n_at(x), M, a) * (m["gt"] * t_at(y)[0][0] * t_at(y)[1][0] + m["ft"])   # noqa: E731
    Tt = lambda x, y: m["gt"] / dt * X(t_at(y), N, b) * (m["gn"] * n_at(x)[0][0] * n_at(x)[1][0] + m["fn"])   # noqa: E731
    Dnn = lambda x, y: m["gn"] / dn ** 2 * Z(n_at(x), M, a) * (m["gt"] * t_at(y)[0][0] * t_at(y)[1][0] + m["ft"])  # noqa: E731
    Dtt = lambda x, y: m["gt"] / dt ** 2 * Z(t_at(y), N, b) * (m["gn"] * n_at(x)[0][0] * n_at(x)[1][0] + m["fn"])  # noqa: E731
    Dnt = lambda x, y: m["gn"] * m["gt"] / dn / dt * X(n_at(x), M, a) * X(t_at(y), N, b)                        # noqa: E731
    zero = torch.zeros_like(opn)
    contact = opn < 0
    x = torch.where(contact, zero, opn)          # tangential terms see no opening in contact
    over = (opn > dn) | (opt > dt)
    x, y = torch.where(over, zero, x), torch.where(over, zero, opt)
    tt, tn = Tt(x, y), Tn(x, y)
    eps = -1e-9
    bad = (tt < eps) | ((y > dt * m["lambda_t"] / 5) & (tt < 0.05 * m["tau_max"]))
    bad |= ~contact & ((tn < eps) | ((x > dn * m["lambda_n"] / 5) & (tn < 0.05 * m["sigma_max"])))
    failed = over | bad
    tsoft, nsoft = y >= tmax, (x >= pmax) & ~contact
    safe_p, safe_t = torch.where(pmax > 0, pmax, zero + 1), torch.where(tmax > 0, tmax, zero + 1)
    # normal direction: softening at the present (or largest) tangential opening, else the secant
    peak_n = Tn(pmax, tmax) / safe_p
    dnn0 = Dnn(zero, tmax)
    at = torch.where(tsoft, y, tmax)
    out_n = torch.where(nsoft, Tn(x, at), torch.where(pmax > 0, peak_n * opn, torch.where(contact, dnn0 * opn, zero)))
    out_dnn = torch.where(nsoft, Dnn(x, at), torch.where(pmax > 0, peak_n, dnn0))
    # tangential direction: at zero normal opening in contact, at the larger of history and present else
    ref = torch.where(contact, zero, torch.where(nsoft & tsoft, x, pmax))
    peak_t = Tt(ref, tmax) / safe_t
    out_t = torch.where(tsoft, Tt(ref, y), torch.where(tmax > 0, peak_t * opt, zero))
    out_dtt = torch.where(tsoft, Dtt(ref, y), torch.where(tmax > 0, peak_t, Dtt(ref, zero)))
    out_dnt = torch.where(tsoft & nsoft, Dnt(x, y), zero)
    keep = ~failed
    z = [torch.where(keep, v, zero) for v in (out_n, out_t, out_dnn, out_dtt, out_dnt)]
    pm = torch.where(keep & nsoft, opn, pmax)
    tm = torch.where(keep & tsoft, opt, tmax)
    return z, pm, tm, failed


def _assembled(col, czs, un, vn, an, pmax, tmax, cs, blocks):
    """Tangent values (room for `blocks` of them), residual rows, node forces and CZ records (stride
    cs) of one iteration."""
    m = _material()
    alt, N, keys = _pattern(col, czs)
    dev = alt.device
    f64 = lambda v: torch.as_tensor(np.ascontiguousarray(v), dtype=torch.float64, device=dev)   # noqa: E731
    x0, un, vn, an = f64(col.x0), f64(un), f64(vn), f64(an)
    n, ns = len(x0), stride_of(len(x0))
    vals = torch.zeros(max(blocks, keys.numel()), 9, dtype=torch.float64, device=dev)
    rhs = torch.zeros(N, 3, dtype=torch.float64, device=dev)
    F = torch.zeros(n, 3, dtype=torch.float64, device=dev)
    stiff = 1 + m["dampingStiffness"] * GAMMA / (H * BETA)
    mcoef = (1 / H ** 2 + m["dampingMass"] * GAMMA / H) / BETA
    eye = torch.eye(3, dtype=torch.float64, device=dev)

    def add(units, i, j, block):
        p, q = alt[units[:, i]], alt[units[:, j]]
        ok = (p >= 0) & (q >= p)
        vals.index_add_(0, torch.searchsorted(keys, (p * N + q)[ok]), block.reshape(-1, 9)[ok])

    def add_rows(units, i, r):
        p = alt[units[:, i]]
        rhs.index_add_(0, p[p >= 0], r[p >= 0])

    for part in torch.as_tensor(col.elastic, device=dev).split(200_000):
        X = x0[part]
        x = X + un[part]
        p, q, r = (X[:, 1:] - X[:, :1]).unbind(1)
        g = torch.stack([torch.linalg.cross(q, r), torch.linalg.cross(r, p), torch.linalg.cross(p, q)], 1)
        det = (p * g[:, 0]).sum(-1)
        V = det / 6
        g = g / det[:, None, None]
        g = torch.cat([-g.sum(1, keepdim=True), g], 1)                              # (T, 4, 3)
        R = _times(_frame(*x[:, :3].unbind(1)), _frame(*X[:, :3].unbind(1)).transpose(1, 2))
        G = _times(g, R.transpose(1, 2))                                            # rotated gradients
        gg = (G[:, :, None] * G[:, None]).sum(-1)
        outer = G[:, :, None, :, None] * G[:, None, :, None, :]                     # (T, i, j, k, l)
        K = V[:, None, None, None, None] * (m["lam"] * outer + m["mu"] * outer.transpose(3, 4)
                                            + m["mu"] * gg[..., None, None] * eye)
        mass = m["rho"] / 20 * (1 + torch.eye(4, dtype=torch.float64, device=dev))
        y = x - _times(X, R.transpose(1, 2)) + m["dampingStiffness"] * vn[part]            # R (R^T x - x0) + damping
        q = m["dampingMass"] * vn[part] + an[part]
        r = -(K * y[:, None, :, None, :]).sum((2, 4)) - V[:, None, None] * (mass @ q)
        r[..., 2] += (m["gravity"] * m["rho"] * V / 4)[:, None]
        lhs = stiff * K + mcoef * V[:, None, None, None, None] * mass[None, :, :, None, None] * eye
        for i in range(4):
            F.index_add_(0, part[:, i], r[:, i])
            add_rows(part, i, r[:, i])
            for j in range(4):
                add(part, i, j, lhs[:, i, j])
    C = len(czs)
    dcz = torch.zeros(10, cs, dtype=torch.float64, device=dev)
    units = torch.as_tensor(czs, device=dev)
    x = (x0 + un)[units]
    mid = (x[:, :3] + x[:, 3:]) / 2
    e1 = torch.nn.functional.normalize(mid[:, 1] - mid[:, 0], dim=-1)
    w = torch.linalg.cross(mid[:, 1] - mid[:, 0], mid[:, 0] - mid[:, 2])
    nv = torch.nn.functional.normalize(w, dim=-1)
    R = torch.stack([e1, torch.linalg.cross(nv, e1), nv], 1)                        # rows
    area = w.norm(dim=-1) / 2
    gp = torch.tensor([[1 / 6, 2 / 3], [2 / 3, 1 / 6], [1 / 6, 1 / 6]], dtype=torch.float64, device=dev)
    sf = torch.stack([1 - gp.sum(1), gp[:, 0], gp[:, 1]])                           # (node, gp)
    gap = _times(_times(x[:, :3] - x[:, 3:], R.transpose(1, 2)).transpose(1, 2), sf)   # (C, direction, gp)
    d1, d2, opn = gap.unbind(1)
    opt = (d1 * d1 + d2 * d2).sqrt()
    (Tn, Tt, Dnn, Dtt, Dnt), pm, tm, fail = _law(m, opn, opt, f64(pmax), f64(tmax))
    failed = fail.any(1)
    o = torch.where(opt < 1e-20, torch.ones_like(opt), opt)
    c, s = d1 / o, d2 / o
    tr = torch.stack([Tt * c, Tt * s, Tn], 1)                                       # (C, 3, gp)
    Td = torch.stack([Dtt * c * c + Tt * s * s / o, (Dtt - Tt / o) * c * s, Dnt * c,
                      (Dtt - Tt / o) * c * s, Dtt * s * s + Tt * c * c / o, Dnt * s,
                      Dnt * c, Dnt * s, Dnn], -1).reshape(C, 3, 3, 3)               # (C, gp, 3, 3)
    wa = torch.where(failed, torch.zeros_like(area), area / 3)
    Tg = _times(R.transpose(1, 2), tr) * wa[:, None, None]
    Q = _times(_times(R.transpose(1, 2)[:, None], Td), R[:, None]) * wa[:, None, None, None]
    for a in range(6):
        sa = 1 if a < 3 else -1
        add_rows(units, a, -sa * (Tg * sf[a % 3]).sum(-1))
        for b in range(6):
            sb = sa if b < 3 else -sa
            add(units, a, b, sb * (Q * (sf[a % 3] * sf[b % 3])[None, :, None, None]).sum(1))
    dcz[0:3, :C], dcz[3:6, :C] = pm.max(1).values, tm.max(1).values
    ok = ~failed
    for k, v in enumerate((opn, opt, Tn, Tt)):
        dcz[6 + k, :C] = torch.where(ok, v.mean(1), torch.zeros_like(area))
    out = torch.zeros(3, ns, dtype=torch.float64, device=dev)
    out[:, :n] = F.T
    return dict(vals=vals.reshape(-1), rhs=rhs.reshape(-1), F=out.reshape(-1), dcz=dcz.reshape(-1),
                flags=None)


def exact(case, seed):
    """Tangent, residual, forces and CZ records of a first pass; none for the cases with contact,
    whose values hang on the impacts that detection finds."""
    if case["kind"] in ("contact", "replay"):
        return None
    col = _mesh_of(case)
    _, s, du, _ = _state(case, col, seed)
    czs, pmax, tmax, C = col.czs, s.pmax, s.tmax, len(col.czs)
    if case["kind"] == "dropin":
        un, vn, an = s.un, s.vn, s.an
    else:
        un = (s.un - du) + du
        an = s.an * (1 - 1 / (2 * BETA)) + du / (H * H * BETA) - s.vn / (H * BETA)
        vn = s.vn + H * ((1 - GAMMA) * s.an + GAMMA * an)
    blocks = 0
    if case["kind"] == "fracture":
        blocks = _pattern(col, czs)[2].numel()
        first = max(1, C // 50)
        czs, pmax, tmax = czs[first:], pmax[first:], tmax[first:]
    out = _assembled(col, czs, un, vn, an, pmax, tmax, stride_of(C), blocks)
    if case["kind"] == "batched":
        out["counts"] = [None, None]
    else:
        out["counts"] = [None] * (2 if case["kind"] == "dropin" else 4)
    if case["kind"] == "fracture":
        out.update(rows=None, cols=None)
    return out
