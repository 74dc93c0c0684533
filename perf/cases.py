"""The work a program has this framework do, as cases that can be timed.

A case is one of these jobs on a mesh of the unit square (P1 or P2 triangles)
or the unit cube (P1 tetrahedra) whose interior vertices are jittered by the
seed:

  system      assemble an operator, discretise the right-hand side and
              eliminate the boundary DOFs (what precedes every solve)
  errors      L2 and H1 error of a finite element function (what follows it)
  products    A x and A^T x with the assembled CSR matrix
  pcg         FP64 CG to a relative residual of 1e-10 with an FP32 or an FP64
              V-cycle on a hierarchy that the program keeps
  stationary  AMGSolver::solve with its default arguments (21 FP64 V(3,3)
              cycles on the hierarchy of AMGSolver(A))
  moving      one step of a moving mesh: new coordinates, system, values-only
              refresh of the hierarchy, solve
  batch       uneven problems solved together by the continuous batch

Vectors live in torch tensors on the GPU; the library takes their pointers.
exact() restates the same job in plain torch FP64: numbering, pattern,
quadrature, elimination and a Jacobi CG to a residual of 1e-13.
"""
import ctypes
import math

import numpy as np
import torch

import afepack_amd as afe

P1, P2, TET = afe.P1_TRI, afe.P2_TRI, afe.P1_TET
OPS = {"stiff": afe.OP_STIFF, "mass": afe.OP_MASS, "var": afe.OP_VARSTIFF}
RHS = {"poisson": afe.F_POISSON, "varcoef": afe.F_VARCOEF, "nodal": afe.F_NODAL, "one": afe.F_ONE}

# The sizes are those of the benchmark's workloads (64^2 P1, 1024^2 P2, 3D P1
# with a 16-mode coefficient, uneven 2D problems with n in [32, 512], serving
# requests of 1e3 to 2e6 DOFs) and odd sizes between them.


def listed():
    return [
        # the reference's first example: latency of three short calls
        dict(name="system p1 64", job="system", kind=P1, n=64, acc=4, op="stiff", rhs="poisson"),
        # the benchmark's large 2D system
        dict(name="system p2 1024", job="system", kind=P2, n=1024, acc=6, op="stiff", rhs="poisson"),
        # an odd-sized problem of the uneven batch: 8-mode coefficient, load given at the DOFs
        dict(name="system p2 301 var", job="system", kind=P2, n=301, acc=6, op="var", rhs="nodal"),
        # the 3D variable-coefficient problem with its manufactured load
        dict(name="system tet 80 var", job="system", kind=TET, n=80, acc=2, op="var", rhs="varcoef"),
        # error control after a 2M-DOF solve
        dict(name="errors p2 701", job="errors", kind=P2, n=701, acc=6),
        # SparseMatrix::vmult and Tvmult in a caller's own iteration
        dict(name="products p2 512", job="products", kind=P2, n=512, acc=6, op="stiff"),
        # the reference's solver with its defaults at the size of its example
        dict(name="stationary p1 64", job="stationary", kind=P1, n=64, acc=4),
        # a single mid-size solve (a serving request)
        dict(name="pcg p2 256", job="pcg", kind=P2, n=256, acc=6, op="stiff", rhs="poisson", prec="fp32",
             nmpo=50, smooth=1),
        # the benchmark's headline solve
        dict(name="pcg p2 1024", job="pcg", kind=P2, n=1024, acc=6, op="stiff", rhs="poisson", prec="fp32",
             nmpo=2048, smooth=1),
        # a 3D solve with the FP64 V-cycle
        dict(name="pcg tet 71 fp64", job="pcg", kind=TET, n=71, acc=2, op="var", rhs="varcoef", prec="fp64",
             nmpo=50, smooth=1),
        # a moving-mesh re-solve (two of five serving requests)
        dict(name="moving p1 500", job="moving", kind=P1, n=500, acc=4, op="stiff", rhs="poisson", nmpo=50,
             smooth=1),
        # problems of the uneven batch
        dict(name="batch 16", job="batch", count=16, lo=32, hi=256, mix=1, smooth=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    job = rng.choice(["system", "system", "errors", "products", "stationary", "pcg", "pcg", "moving", "batch"])
    if job == "batch":
        return dict(job=job, count=rng.randint(2, 20), lo=32, hi=_log_int(rng, 64, 256), mix=rng.randint(1, 1 << 20),
                    smooth=rng.randint(1, 2))
    if job == "stationary":
        return dict(job=job, kind=P1, n=_log_int(rng, 16, 160), acc=4)
    kind = rng.choice([P1, P2, TET])
    acc = {P1: 4, P2: 6, TET: 2}[kind]
    top = {P1: 1000, P2: 600, TET: 80}[kind]
    if job in ("pcg", "moving"):
        top = {P1: 700, P2: 400, TET: 64}[kind]
    n = _log_int(rng, {P1: 24, P2: 12, TET: 8}[kind], top)
    c = dict(job=job, kind=kind, n=n, acc=acc)
    if job == "errors":
        return c
    if job == "products":
        return dict(c, op="stiff")
    if job == "system":
        op = rng.choice(["stiff", "mass", "var"])
        rhs = {"stiff": "poisson", "mass": rng.choice(["nodal", "one"]), "var": rng.choice(["nodal", "varcoef"])}[op]
        return dict(c, op=op, rhs=rhs)
    op, rhs = rng.choice([("stiff", "poisson"), ("var", "varcoef"), ("var", "nodal")])
    c = dict(c, op=op, rhs=rhs, nmpo=50 if job == "moving" else rng.choice([50, 512]), smooth=rng.randint(1, 2))
    return c if job == "moving" else dict(c, prec=rng.choice(["fp32", "fp64"]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _mesh(kind, n, rng):
    """coords (n_vert, dim), elem_vert (n_elem, dim + 1), vert_mark: squares split along one diagonal, row by
    row, or cubes into six tetrahedra; interior vertices jittered (0.2 h in 2D, 0.05 h in 3D)"""
    if kind == TET:
        g = np.arange(n + 1)
        x, y, z = np.meshgrid(g, g, g, indexing="ij")
        co = np.stack([x.ravel(), y.ravel(), z.ravel()], 1)
        split = np.array([[0, 1, 4, 2], [4, 2, 1, 5], [3, 2, 5, 1], [4, 6, 2, 5], [3, 6, 5, 2], [7, 6, 5, 3]])
        off = np.array([(c >> 2) * (n + 1) ** 2 + (c >> 1 & 1) * (n + 1) + (c & 1) for c in range(8)])
        i, j, k = np.meshgrid(np.arange(n), np.arange(n), np.arange(n), indexing="ij")
        base = ((i * (n + 1) + j) * (n + 1) + k).ravel()
        ev = (base[:, None, None] + off[split][None]).reshape(-1, 4)
        jitter = 0.05
    else:
        y, x = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
        co = np.stack([x.ravel(), y.ravel()], 1)
        j, i = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
        a = (j * (n + 1) + i).ravel()
        ev = np.stack([a, a + 1, a + n + 2, a, a + n + 2, a + n + 1], 1).reshape(-1, 3)
        jitter = 0.2
    edge = ((co == 0) | (co == n)).any(1)
    pts = co / n
    pts += np.where(edge[:, None], 0.0, rng.uniform(-jitter / n, jitter / n, pts.shape))
    return pts, ev.astype(np.int32), edge.astype(np.int32)


def _field(kind, rng):
    """the coefficient a = exp(g): 8 modes of amplitude 0.5 in 2D, 16 of amplitude 1 in 3D, wave numbers 1 to 4"""
    m, dim, amp = (16, 3, 1.0) if kind == TET else (8, 2, 0.5)
    w = rng.uniform(0.5, 1.0, m)
    s = amp / w.sum()
    return dict(k=rng.integers(1, 5, (m, dim)).astype(float), phi=rng.uniform(0, 2 * math.pi, m),
                w=w * rng.choice([-1.0, 1.0], m), scale=s)


def _inputs(case, seed):
    rng = np.random.default_rng([int(seed), case["kind"], case["n"]])
    n_dof = _n_dof(case)
    co, ev, vm = _mesh(case["kind"], case["n"], rng)
    inp = dict(co=co, ev=ev, vm=vm, field=_field(case["kind"], rng))
    if case.get("rhs") == "nodal":
        inp["nodal"] = rng.uniform(-1.0, 1.0, n_dof)
    if case["job"] == "products":
        inp["x"], inp["xt"] = rng.standard_normal(n_dof), rng.standard_normal(n_dof)
    if case["job"] == "errors":
        inp["noise"] = rng.uniform(-1e-3, 1e-3, n_dof)
    if case["job"] == "moving":
        k = int(rng.integers(1, 4))
        inner = (vm == 0)[:, None]
        inp["moved"] = co + np.where(inner, 0.1 / case["n"] * np.sin(2 * math.pi * k * co), 0.0)
    return inp


def _members(case, seed):
    """the problems of a batch: P1 and P2 in turn, n log-uniform (drawn by the case's mix), each its own mesh, field
    and load"""
    rng = np.random.default_rng(case["mix"])
    n = np.rint(np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["count"]))).astype(int)
    return [(dict(job="pcg", kind=P1 if i % 2 == 0 else P2, n=int(m), acc=4 if i % 2 == 0 else 6, op="var",
                  rhs="nodal"), int(seed) * 1000 + i) for i, m in enumerate(n)]


# ---------------------------------------------------------------------------
# the framework's objects, as a program that keeps its vectors in torch has them
# ---------------------------------------------------------------------------
class _Vector(afe.DeviceVector):
    """a torch tensor handed to the library by its pointer"""

    def __init__(self, ctx, tensor):
        self.ctx, self.tensor = ctx, tensor.contiguous()
        self.n, self.dtype = tensor.numel(), np.dtype(np.float64)
        self.nbytes = 8 * self.n
        self.ptr = ctypes.c_void_p(self.tensor.data_ptr())

    def free(self):
        self.ptr = None


class _Values:
    """the device values of a matrix as a torch tensor that keeps the matrix alive"""

    def __init__(self, matrix):
        self.matrix = matrix
        ptr = afe.load().afe_matrix_device_values(matrix.h)
        self.__cuda_array_interface__ = dict(shape=(matrix.nnz,), typestr="<f8", data=(ptr, False), version=2)


_context = []


def _ctx():
    if not _context:
        _context.append(afe.Context(0))
    return _context[0]


def _vec(a):
    return _Vector(_ctx(), torch.as_tensor(a, dtype=torch.float64).cuda())


def _zeros(n):
    return _Vector(_ctx(), torch.zeros(n, dtype=torch.float64, device="cuda"))


def _build_system(s):
    """operator, right-hand side and boundary elimination into s's matrix and load"""
    c = s["case"]
    s["A"].assemble(OPS[c["op"]], c["acc"], s["field"] if c["op"] == "var" else None)
    s["sp"].rhs(c["acc"], RHS[c["rhs"]], s["field"] if c["rhs"] == "varcoef" else None, nodal=s.get("nodal"), out=s["f"])
    if c["op"] != "mass":
        s["A"].apply_dirichlet(s["f"])


def _problem(case, seed):
    inp = _inputs(case, seed)
    sp = afe.Space(_ctx(), case["kind"], inp["co"].ravel(), inp["ev"].ravel(), inp["vm"])
    f = inp["field"]
    s = dict(case=case, sp=sp, field=afe.Field(f["k"].ravel(), f["phi"], f["w"], f["scale"]), inp=inp)
    if "nodal" in inp:
        s["nodal"] = _vec(inp["nodal"])
    if case["job"] != "errors":
        s["A"] = afe.Matrix(sp)
        s["values"] = torch.as_tensor(_Values(s["A"]), device="cuda")
        s["f"] = _zeros(sp.n_dof)
    return s


def prepare(case, seed):
    job = case["job"]
    if job == "batch":
        members = [_problem(c, sd) for c, sd in _members(case, seed)]
        for s in members:
            _build_system(s)
            s["g"] = afe.Amg(s["A"], afe.AmgParams(lazy=1, smooth=case["smooth"], build_fp32=1))
            s["x"] = _zeros(s["sp"].n_dof)
        state = dict(case=case, members=members)
    elif job == "errors":
        state = _problem(case, seed)
        p = state["sp"].dofs()[2].reshape(-1, state["sp"].dim)
        state["uh"] = _vec(np.sin(math.pi * p).prod(1) + state["inp"]["noise"])
    elif job == "products":
        state = _problem(case, seed)
        state["A"].assemble(OPS[case["op"]], case["acc"])
        n = state["sp"].n_dof
        state.update(x=_vec(state["inp"]["x"]), xt=_vec(state["inp"]["xt"]), y=_zeros(n), yt=_zeros(n))
    else:
        if job == "stationary":
            case = dict(case, op="stiff", rhs="poisson")
        state = _problem(case, seed)
        if job != "system":
            _build_system(state)
            if job == "stationary":
                prm = afe.AmgParams()
            else:
                prm = afe.AmgParams(lazy=1, nmpo=case["nmpo"], nmpsd=0.382 if case["nmpo"] == 50 else 0.0,
                                    smooth=case["smooth"], build_fp32=1)
            state["g"] = afe.Amg(state["A"], prm)
            state["x"] = _zeros(state["sp"].n_dof)
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    job = case["job"]
    if job == "system":
        _build_system(state)
        return dict(values=state["values"], f=state["f"].tensor)
    if job == "errors":
        return [state["sp"].error_l2(state["uh"], case["acc"]), state["sp"].error_h1(state["uh"], case["acc"])]
    if job == "products":
        state["A"].vmult(state["x"], state["y"])
        state["A"].tvmult(state["xt"], state["yt"])
        return [state["y"].tensor, state["yt"].tensor]
    if job == "batch":
        batch = afe.Batch(_ctx(), afe.PREC_FP32, smooth=case["smooth"])
        for s in state["members"]:
            s["x"].zero()
            batch.add(s["g"], s["x"], s["f"], rtol=1e-10, max_it=1000)
        batch.run()
        batch.close()
        return [s["x"].tensor for s in state["members"]]
    x = state["x"]
    if job == "moving":
        state["sp"].update_coords(state["inp"]["moved"].ravel())
        _build_system(state)
        state["g"].lazy_reinit(state["A"])
    x.zero()
    if job == "stationary":
        state["g"].solve(x, state["f"])
    else:
        prec = afe.PREC_FP64 if case.get("prec") == "fp64" else afe.PREC_FP32
        state["g"].pcg(x, state["f"], rtol=1e-10, max_it=1000, prec=prec)
    if job == "moving":
        return dict(values=state["values"], x=x.tensor)
    return x.tensor


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _n_dof(case):
    k, n = case["kind"], case["n"]
    return (n + 1) ** 3 if k == TET else (2 * n + 1) ** 2 if k == P2 else (n + 1) ** 2


def _sizes(case):
    """DOFs, matrix entries, vertices, elements, local DOFs, vertices per element, dimension, quadrature points"""
    k, n = case["kind"], case["n"]
    if k == TET:
        return (n + 1) ** 3, 15 * n ** 3 + 21 * n ** 2 + 9 * n + 1, (n + 1) ** 3, 6 * n ** 3, 4, 4, 3, 4
    nnz = 46 * n * n + 16 * n + 1 if k == P2 else 7 * n * n + 6 * n + 1
    return _n_dof(case), nnz, (n + 1) ** 2, 2 * n * n, 6 if k == P2 else 3, 3, 2, 12 if k == P2 else 6


def work(case):
    job = case["job"]
    if job == "batch":
        parts = [work(dict(c, prec="fp32", nmpo=50, smooth=case["smooth"])) for c, _ in _members(case, 1)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    m, nnz, nv, ne, nl, nvx, dim, nq = _sizes(case)
    mesh = nv * dim * 8 + ne * (nvx + nl) * 4  # coordinates, element vertices and DOFs
    point = 2 * nl * dim + 6 * dim * dim + 10  # basis and mapping at one quadrature point
    trig = (16 if dim == 3 else 8) * (2 * dim + 20)  # the coefficient there: one sine per mode
    if job == "errors":
        return {"bytes": 2.0 * (mesh + m * 8), "flops": 2.0 * ne * nq * (point + 30 * dim)}
    if job == "products":
        return {"bytes": 2.0 * (nnz * 12 + m * 20), "flops": 4.0 * nnz}
    op, rhs = case.get("op", "stiff"), case.get("rhs", "poisson")
    sysb = 2 * mesh + nnz * 8 + m * 8 + (m * 8 if rhs == "nodal" else 0)
    if op != "mass":  # the elimination reads the pattern and marks and rewrites the rows it changes
        sysb += m * 12
    sysf = ne * nq * (2 * point + nl * (nl + 1) // 2 * (2 * dim + 2) + 3 * nl)
    sysf += ne * nq * trig * ((op == "var") + (rhs == "varcoef"))
    if job == "system":
        return {"bytes": float(sysb), "flops": float(sysf)}
    if job == "stationary":  # 21 cycles of six sweeps, the residual and the transfers over levels that add a quarter
        return {"bytes": 21 * 7.0 * 1.25 * (nnz * 12 + 3 * m * 8), "flops": 21 * 7 * 1.25 * 2.0 * nnz}
    # CG: the iterations these systems take, each one FP64 product, one V-cycle and the vector updates
    its = {P1: 12 + 3 * math.log2(max(case["n"], 16) / 16), P2: 28 + 6 * math.log2(max(case["n"], 32) / 32), TET: 18}
    sv = 8 if case.get("prec") == "fp64" else 4
    its = its[case["kind"]]
    b = its * (nnz * 12 + m * 16 + 1.2 * (2 * case["smooth"] + 1) * (nnz * (sv + 4) + 3 * m * sv) + 13 * m * 8)
    f = its * (2.0 * nnz + 1.2 * (2 * case["smooth"] + 1) * 2 * nnz + 10 * m)
    if job == "moving":
        b, f = b + sysb + nnz * 24, f + sysf + 2.0 * nnz
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# the same jobs in plain torch FP64
# ---------------------------------------------------------------------------
_D = torch.float64


def _rule(kind, acc):
    """barycentric points and weights of the reference's rules of these accuracies"""
    if kind == TET:  # accuracy 2, 4 points
        assert acc == 2
        a, b = 0.58541020, 0.13819660
        p = [(b, b, b), (a, b, b), (b, a, b), (b, b, a)]
        return torch.tensor([(1 - sum(q),) + q for q in p], dtype=_D, device="cuda"), [0.25] * 4
    if acc == 4:  # 6 points
        g = [((0.108103018168070, 0.445948490915965, 0.445948490915965), 0.223381589678011),
             ((0.816847572980459, 0.091576213509771, 0.091576213509771), 0.109951743655322)]
        orders = [(0, 1, 2), (1, 2, 0), (2, 0, 1)]
        p = [(tuple(t[o] for o in od), w) for t, w in g for od in orders]
    else:  # accuracy 6, 12 points
        assert acc == 6
        g = [((0.501426509658179, 0.249286745170910, 0.249286745170910), 0.116786275726379),
             ((0.873821971016996, 0.063089014491502, 0.063089014491502), 0.050844906370207)]
        p = [(tuple(t[o] for o in od), w) for t, w in g for od in [(0, 1, 2), (1, 2, 0), (2, 0, 1)]]
        t, w = (0.053145049844817, 0.310352451033784, 0.636502499121399), 0.082851075618374
        p += [(tuple(t[o] for o in od), w) for od in [(0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)]]
    lam = torch.tensor([(1 - q[1] - q[2], q[1], q[2]) for q, _ in p], dtype=_D, device="cuda")
    return lam, [w for _, w in p]


class _Exact:
    """mesh, numbering, pattern and element geometry of a case on the GPU"""

    def __init__(self, case, inp, coords=None):
        self.case, self.kind = case, case["kind"]
        self.co = torch.as_tensor(inp["co"] if coords is None else coords, dtype=_D).cuda()
        ev = torch.as_tensor(inp["ev"]).long().cuda()
        self.ev = ev
        vm = torch.as_tensor(inp["vm"]).cuda() != 0
        ne, nvx = ev.shape
        key = ev
        if self.kind == P2:  # edges opposite each vertex, numbered behind the vertices
            a, b = ev[:, [1, 2, 0]], ev[:, [2, 0, 1]]
            ek = torch.minimum(a, b) * len(vm) + torch.maximum(a, b)
            _, inv, cnt = torch.unique(ek, return_inverse=True, return_counts=True)
            key = torch.cat([ev, inv + len(vm)], 1)
            mark = torch.cat([vm, cnt == 1])
        else:
            mark = vm
        # DOFs are numbered on first touch, element by element
        flat = key.reshape(-1)
        ids, inv = torch.unique(flat, return_inverse=True)
        first = torch.full((len(ids),), flat.numel(), dtype=torch.int64, device="cuda")
        first.scatter_reduce_(0, inv, torch.arange(flat.numel(), device="cuda"), "amin")
        order = torch.argsort(first)
        rank = torch.empty_like(order)
        rank[order] = torch.arange(len(order), device="cuda")
        self.dof = rank[inv].reshape(key.shape)
        self.n = len(ids)
        self.mark = mark[ids][order]
        self.nl = key.shape[1]
        v = self.co[ev]
        e = v[:, 1:] - v[:, :1]
        self.v = v
        self.det = torch.linalg.det(e) if self.kind == TET else e[:, 0, 0] * e[:, 1, 1] - e[:, 0, 1] * e[:, 1, 0]
        inv_t = torch.linalg.inv(e) if self.kind == TET else torch.stack(
            [torch.stack([e[:, 1, 1], -e[:, 0, 1]], 1), torch.stack([-e[:, 1, 0], e[:, 0, 0]], 1)], 1) / self.det[:, None, None]
        g = inv_t.transpose(1, 2)  # row i: gradient of barycentric i + 1
        self.dl = torch.cat([-g.sum(1, keepdim=True), g], 1)
        self.vol = self.det / (6.0 if self.kind == TET else 2.0)
        self.lam, self.w = _rule(self.kind, case["acc"])

    def basis(self, q):
        la = self.lam[q]
        if self.kind != P2:
            return la
        a, b, c = la
        return torch.stack([a * (2 * a - 1), b * (2 * b - 1), c * (2 * c - 1), 4 * b * c, 4 * a * c, 4 * a * b])

    def grads(self, q):
        if self.kind != P2:
            return self.dl
        la, d = self.lam[q], self.dl
        vert = (4 * la - 1)[None, :, None] * d
        edge = 4 * (la[[1, 2, 0]][None, :, None] * d[:, [2, 0, 1]] + la[[2, 0, 1]][None, :, None] * d[:, [1, 2, 0]])
        return torch.cat([vert, edge], 1)

    def at(self, q):
        return (self.lam[q][None, :, None] * self.v).sum(1)

    def coef(self, field, x, grad=False):
        g = torch.zeros(len(x), dtype=_D, device="cuda")
        dg = torch.zeros_like(x)
        for k, phi, w in zip(field["k"], field["phi"], field["w"]):
            kk = torch.tensor(2 * math.pi * k, dtype=_D, device="cuda")
            arg = x @ kk + phi
            g += w * torch.sin(arg)
            if grad:
                dg += (w * torch.cos(arg))[:, None] * kk
        return field["scale"] * g, field["scale"] * dg

    def pattern(self):
        i = self.dof[:, :, None].expand(-1, -1, self.nl).reshape(-1)
        j = self.dof[:, None, :].expand(-1, self.nl, -1).reshape(-1)
        keys, self.inv = torch.unique(i * self.n + j, return_inverse=True)
        self.row, self.col = keys // self.n, keys % self.n
        lead = torch.where(self.row == self.col, torch.zeros_like(self.col), self.col + 1)
        self.order = torch.argsort(self.row * (self.n + 1) + lead)  # diagonal first, the rest ascending

    def matrix(self, op, field):
        self.pattern()
        K = torch.zeros(len(self.det), self.nl, self.nl, dtype=_D, device="cuda")
        for q, w in enumerate(self.w):
            jw = w * self.vol
            if op == "mass":
                b = self.basis(q)
                K += jw[:, None, None] * (b[:, None] * b[None, :])
                continue
            if op == "var":
                jw = jw * torch.exp(self.coef(field, self.at(q))[0])
            g = self.grads(q)
            K += jw[:, None, None] * (g @ g.transpose(1, 2).contiguous() if self.kind == TET else
                                      g[:, :, None, 0] * g[:, None, :, 0] + g[:, :, None, 1] * g[:, None, :, 1])
        val = torch.zeros(len(self.row), dtype=_D, device="cuda")
        return val.index_add_(0, self.inv, K.reshape(-1))

    def load(self, rhs, field, nodal):
        f = torch.zeros(self.n, dtype=_D, device="cuda")
        dim = self.co.shape[1]
        for q, w in enumerate(self.w):
            x, b = self.at(q), self.basis(q)
            if rhs == "one":
                s = torch.ones(len(x), dtype=_D, device="cuda")
            elif rhs == "nodal":
                s = torch.as_tensor(nodal).cuda()[self.dof] @ b
            else:
                s = dim * math.pi ** 2 * torch.sin(math.pi * x).prod(1)
                if rhs == "varcoef":
                    g, dg = self.coef(field, x, True)
                    s = torch.exp(g) * (s - (dg * self.grad_u(x)).sum(1))
            f.index_add_(0, self.dof.reshape(-1), ((w * self.vol * s)[:, None] * b[None]).reshape(-1))
        return f

    @staticmethod
    def grad_u(x):
        s, c = torch.sin(math.pi * x), math.pi * torch.cos(math.pi * x)
        return torch.stack([c[:, d] * torch.cat([s[:, :d], s[:, d + 1:]], 1).prod(1) for d in range(x.shape[1])], 1)

    def system(self, inp):
        c = self.case
        val = self.matrix(c["op"], inp["field"])
        f = self.load(c["rhs"], inp["field"], inp.get("nodal"))
        if c["op"] != "mass":
            out = (self.mark[self.row] | self.mark[self.col]) & (self.row != self.col)
            val[out] = 0.0
            f[self.mark] = 0.0
        return val, f

    def solve(self, val, f):
        crow = torch.zeros(self.n + 1, dtype=torch.int64, device="cuda")
        crow[1:] = torch.cumsum(torch.bincount(self.row, minlength=self.n), 0)
        A = torch.sparse_csr_tensor(crow, self.col, val, (self.n, self.n))
        dinv = 1.0 / val[self.row == self.col]
        x, r = torch.zeros_like(f), f.clone()
        z = dinv * r
        p, rz = z.clone(), r @ z
        for it in range(20000):
            q = A @ p
            a = rz / (p @ q)
            x.addcmul_(a, p)
            r.addcmul_(a, q, value=-1)
            torch.mul(dinv, r, out=z)
            new = r @ z
            p.mul_(new / rz).add_(z)
            rz = new
            if it % 50 == 49 and float(r.norm()) <= 1e-13 * float(f.norm()):
                break
        return x


def exact(case, seed):
    job = case["job"]
    if job == "stationary":  # a fixed number of cycles: not the solution itself
        return None
    if job == "batch":
        out = []
        for c, sd in _members(case, seed):
            inp = _inputs(c, sd)
            e = _Exact(c, inp)
            out.append(e.solve(*e.system(inp)))
        return out
    if job in ("pcg", "moving") and _n_dof(case) > 1500000:  # the plain CG takes too long
        return None
    inp = _inputs(case, seed)
    e = _Exact(case, inp, inp.get("moved"))
    if job == "errors":
        dof_co = torch.zeros(e.n, e.co.shape[1], dtype=_D, device="cuda")
        pts = e.v if e.kind != P2 else torch.cat([e.v, 0.5 * (e.v[:, [1, 2, 0]] + e.v[:, [2, 0, 1]])], 1)
        dof_co[e.dof.reshape(-1)] = pts.reshape(-1, e.co.shape[1])
        u = torch.sin(math.pi * dof_co).prod(1) + torch.as_tensor(inp["noise"]).cuda()
        l2 = h1 = 0.0
        for q, w in enumerate(e.w):
            x = e.at(q)
            d = torch.sin(math.pi * x).prod(1) - u[e.dof] @ e.basis(q)
            l2 += float((w * e.vol * d * d).sum())
            g = (u[e.dof][:, :, None] * e.grads(q)).sum(1) - e.grad_u(x)
            h1 += float((w * e.vol * (g * g).sum(1)).sum())
        return [math.sqrt(l2), math.sqrt(h1)]
    if job == "products":
        val = e.matrix(case["op"], inp["field"])
        x, xt = torch.as_tensor(inp["x"]).cuda(), torch.as_tensor(inp["xt"]).cuda()
        y, yt = torch.zeros_like(x), torch.zeros_like(x)
        return [y.index_add_(0, e.row, val * x[e.col]), yt.index_add_(0, e.col, val * xt[e.row])]
    val, f = e.system(inp)
    if job == "system":
        return dict(values=val[e.order], f=f)
    x = e.solve(val, f)
    return dict(values=val[e.order], x=x) if job == "moving" else x
