"""The work that is timed on this framework, through its public entry points.

Each case is one call (or the few calls that belong together) of a program that uses nuto_amd:
assembly of the residual and the tangent, the differentiable residual, batches of meshes, the linear
solve, a load step. `listed` names them, `draw` gives more of the same ranges, `prepare` makes what
the program holds before the call, `run` is the call, `work` what it cannot do without, and `exact`
its outputs from plain torch in 64 bits.

Meshes are bricks of nx x ny x nz cells of 1 mm (tetrahedra: six per brick cell), first-touch dof
numbering. A case is a dict of plain values; the keys that an operation does not use are absent.
"""
import numpy as np
import torch

import nuto_amd as N

NU, E0 = 0.2, 30000.0
MISES_K, KAPPA0, BETA, ALPHA, NONLOCAL_C = 10.0, 1e-4, 100.0, 0.99, 4.0
DECREASING_R, DECREASING_ETA = 0.005, 5.0
DENSITY = 2.4e-9

# element name: (coordinate element, dof element, rule kind, rule order, IPs)
ELEMENTS = {
    "quad4": (N.QUAD4, N.QUAD4, 0, 2, 4),
    "hex8": (N.HEX8, N.HEX8, 0, 2, 8),
    "hex20": (N.HEX8, N.HEX20, 0, 3, 27),
    "tet4": (N.TET4, N.TET4, 1, 1, 1),
    "tet10": (N.TET4, N.TET10, 1, 2, 4),
    "tet10iso": (N.TET10, N.TET10, 1, 2, 4),
}
EDGES = {
    "hex20": ((0, 1), (1, 2), (2, 3), (3, 0), (0, 4), (1, 5), (2, 6), (3, 7), (4, 5), (5, 6), (6, 7), (7, 4)),
    "tet10": ((0, 1), (1, 2), (0, 2), (0, 3), (2, 3), (1, 3)),
}
# a batch lays its element types out in this order
BATCH_ORDER = ("hex20", "tet10", "hex8", "tet4")


def listed():
    return [
        # plane stress, linear elasticity: the smallest full-size workload, a 2D model of 40,000 cells
        dict(name="quad4-plane-stress", op="assemble", element="quad4", law="elastic", nx=200, ny=200, nz=0, jitter=0.0),
        # a mesh of a few hundred cells, as of unit tests, tutorials and material-point studies: latency
        dict(name="hex8-damage-small", op="assemble", element="hex8", law="gradient", nx=7, ny=5, nz=6, jitter=0.0),
        # the headline workload: R + K of gradient damage on a 100 mm cube of a million bricks
        dict(name="hex8-damage-cube", op="assemble", element="hex8", law="gradient", nx=100, ny=100, nz=100, jitter=0.0),
        # the same integrand on a mesh that is not of parallelepipeds, with random material fields
        dict(name="hex8-damage-jittered", op="assemble", element="hex8", law="gradient", nx=59, ny=47, nz=53, jitter=0.1,
             fields=True),
        # the nonlocal interaction that decreases with damage, as structural localisation studies use it
        dict(name="hex8-damage-decreasing", op="assemble", element="hex8", law="gradient", nx=45, ny=43, nz=41, jitter=0.0,
             interaction="decreasing"),
        # identification of material fields: the residual and its gradients with respect to the state and
        # (E, f_t, G_f) through the autograd function
        dict(name="residual-gradient", op="gradient", element="hex8", law="gradient", nx=64, ny=64, nz=64, jitter=0.0,
             fields=True),
        # quadratic bricks, local damage: R + K of a medium model
        dict(name="hex20-damage", op="assemble", element="hex20", law="local", nx=24, ny=23, nz=25, jitter=0.1),
        # a linear elastic analysis on straight-sided quadratic tetrahedra: tangent, then conjugate gradients
        dict(name="tet10-elastic-solve", op="solve", element="tet10", law="elastic", nx=16, ny=15, nz=17, jitter=0.1),
        # one step of an explicit scheme: residual, history update and the stresses to be written, on
        # quadratic tetrahedra with curved edges
        dict(name="tet10-explicit-step", op="explicit", element="tet10iso", law="local", nx=20, ny=21, nz=19, jitter=0.1),
        # many independent meshes of four element types, tuned and replayed (sampling of microstructures)
        dict(name="mixed-batch", op="batch", law="local", meshes=32, lo=1000, hi=20000, jitter=0.1, layout=5),
        # residual, tangent and adjoint of many gradient-damage meshes in one replay
        dict(name="damage-batch-adjoint", op="batch_adjoint", law="gradient", meshes=10, lo=5000, hi=60000, jitter=0.0,
             layout=3),
        # a quasistatic load step of a notched-bar sized model: trial state, Newton without line search, history
        dict(name="load-step", op="load_step", element="hex8", law="gradient", nx=24, ny=8, nz=8, jitter=0.0, fields=True),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    def brick(lo, hi):
        """three different edge lengths around the cube root of a cell count, log-uniform in [lo, hi]"""
        n = size(lo, hi) ** (1.0 / 3.0)
        a, b = rng.uniform(0.75, 1.3), rng.uniform(0.75, 1.3)
        return dict(nx=max(1, round(n * a)), ny=max(1, round(n * b)), nz=max(1, round(n / (a * b))))

    jitter = rng.choice((0.0, 0.1))
    kind = rng.choice(("quad4", "gradient", "gradient", "gradient", "generic", "generic", "explicit", "autograd", "batch",
                       "batch_adjoint", "solve", "load_step"))
    if kind == "quad4":
        return dict(op="assemble", element="quad4", law="elastic", nx=size(4, 400), ny=size(4, 400), nz=0, jitter=jitter,
                    plane=rng.choice(("stress", "strain")))
    if kind == "gradient":
        return dict(op="assemble", element="hex8", law="gradient", jitter=jitter, fields=rng.random() < 0.5,
                    application=rng.choice(("full", "full", "unilateral")),
                    interaction=rng.choice(("constant", "constant", "decreasing")), **brick(100, 150000))
    if kind == "generic":
        element = rng.choice(("hex8", "hex20", "tet4", "tet10", "tet10iso"))
        hi = {"hex8": 100000, "hex20": 13000, "tet4": 40000, "tet10": 20000, "tet10iso": 20000}[element]
        return dict(op="assemble", element=element, law=rng.choice(("elastic", "local")), jitter=jitter,
                    application=rng.choice(("full", "full", "unilateral")), **brick(60, hi))
    if kind == "explicit":
        element = rng.choice(("hex8", "hex20", "tet4", "tet10", "tet10iso"))
        hi = {"hex8": 100000, "hex20": 10000, "tet4": 30000, "tet10": 10000, "tet10iso": 8000}[element]
        return dict(op="explicit", element=element, law="local", jitter=jitter, **brick(60, hi))
    if kind == "autograd":
        return dict(op="gradient", element="hex8", law="gradient", jitter=jitter, fields=True, **brick(200, 260000))
    if kind == "batch":
        return dict(op="batch", law=rng.choice(("local", "elastic")), meshes=rng.randint(4, 32), lo=size(200, 1500),
                    hi=size(3000, 20000), jitter=0.1, layout=rng.randint(1, 10**6))
    if kind == "batch_adjoint":
        return dict(op="batch_adjoint", law="gradient", meshes=rng.randint(2, 10), lo=size(500, 5000),
                    hi=size(8000, 60000), jitter=jitter, layout=rng.randint(1, 10**6))
    if kind == "solve":
        return dict(op="solve", element=rng.choice(("hex8", "tet10")), law="elastic", jitter=0.1, **brick(300, 4000))
    return dict(op="load_step", element="hex8", law="gradient", nx=rng.randint(8, 24), ny=rng.randint(4, 8),
                nz=rng.randint(4, 8), jitter=jitter, fields=True)


# ---- meshes and inputs (numpy, from the seed alone) -----------------------------------------------------------------
def brick_mesh(element, nx, ny, nz, jitter, rng):
    """coordinates (n x dim) and connectivity of a brick of 1 mm cells in the element's node order; every node moved by
    up to jitter mm. tet10iso: nodes at the edge midpoints, moved a little too (curved edges)"""
    ex, ey = nx + 1, ny + 1
    if element == "quad4":
        y, x = np.meshgrid(np.arange(ey), np.arange(ex), indexing="ij")
        X = np.stack([x.ravel() / nx, y.ravel() / ny], 1)  # the unit square
        iy, ix = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
        a = (ix + ex * iy).ravel()
        conn = np.stack([a, a + 1, a + ex + 1, a + ex], 1)
        X = X + rng.uniform(-jitter, jitter, X.shape) * np.array([1.0 / nx, 1.0 / ny])
        return X, conn.astype(np.int32)
    z, y, x = np.meshgrid(np.arange(nz + 1), np.arange(ey), np.arange(ex), indexing="ij")
    X = np.stack([x.ravel(), y.ravel(), z.ravel()], 1).astype(np.float64)
    if jitter:
        X = X + rng.uniform(-jitter, jitter, X.shape)
    iz, iy, ix = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    a = (ix + ex * (iy + ey * iz)).ravel()
    up = ex * ey
    hexa = np.stack([a, a + 1, a + ex + 1, a + ex, a + up, a + up + 1, a + up + ex + 1, a + up + ex], 1)
    if element in ("hex8", "hex20"):
        return X, hexa.astype(np.int32)
    # six tetrahedra around the diagonal 0 - 6
    tets = np.array([[0, 1, 2, 6], [0, 2, 3, 6], [0, 3, 7, 6], [0, 7, 4, 6], [0, 4, 5, 6], [0, 5, 1, 6]])
    conn = hexa[:, tets].reshape(-1, 4)
    if element == "tet10iso":
        ids = entity_ids(conn, EDGES["tet10"], len(X))[:, 4:]
        keys, first, inv = np.unique(ids.ravel(), return_index=True, return_inverse=True)
        ab = conn[:, np.array(EDGES["tet10"])].reshape(-1, 2)[first]
        mid = 0.5 * (X[ab[:, 0]] + X[ab[:, 1]])
        if jitter:
            mid = mid + rng.uniform(-0.2 * jitter, 0.2 * jitter, mid.shape)
        conn = np.concatenate([conn, len(X) + inv.reshape(-1, 6)], 1)
        X = np.concatenate([X, mid])
    return X, conn.astype(np.int32)


def entity_ids(conn, edges, n):
    """per cell: its corner nodes, then one number per edge (the same in every cell that has the edge)"""
    e = np.sort(conn[:, np.array(edges)].astype(np.int64), axis=2)
    return np.concatenate([conn.astype(np.int64), n + e[:, :, 0] * n + e[:, :, 1]], 1)


def batch_meshes(case, seed):
    """[(element, X, conn)]: sizes and types from the case, node positions from the seed"""
    lay = np.random.default_rng(case["layout"])
    out = []
    for m in range(case["meshes"]):
        cells = np.exp(lay.uniform(np.log(case["lo"]), np.log(case["hi"])))
        element = ("tet4", "tet10", "hex8", "hex20")[lay.integers(4)] if case["op"] == "batch" else "hex8"
        bricks = cells / (6.0 if element.startswith("tet") else 1.0)
        n = max(1, round(bricks ** (1.0 / 3.0)))
        nz = max(1, round(bricks / (n * n)))
        out.append((element,) + brick_mesh(element, n, n, nz, case["jitter"], np.random.default_rng([seed, m])))
    return out


def state_arrays(rng, law, dim, nn, n_hist):
    """nodal displacements, nonlocal strains and the history as the damage workloads meet them: undamaged, loading and
    unloading points side by side"""
    amp = 1e-3 if law == "elastic" else 5e-3
    u = rng.uniform(-amp, amp, dim * nn)
    e = rng.uniform(0.0, 5e-4, nn) if law == "gradient" else None
    kappa = None if law == "elastic" else rng.uniform(0.0, 3e-4, n_hist)
    return u, e, kappa


def material_fields(rng, n):
    """E ~ LN(30000, 0.1), f_t ~ LN(3, 0.1), G_f ~ LN(0.1, 0.15) per cell (mean, coefficient of variation)"""
    out = []
    for mean, cv in ((E0, 0.1), (3.0, 0.1), (0.1, 0.15)):
        s2 = np.log1p(cv * cv)
        out.append(np.exp(np.log(mean) - 0.5 * s2 + np.sqrt(s2) * rng.standard_normal(n)))
    return np.stack(out)


def inputs(case, seed):
    """mesh, state and fields of a single-mesh case"""
    rng = np.random.default_rng(seed)
    X, conn = brick_mesh(case["element"], case["nx"], case["ny"], case["nz"], case["jitter"], rng)
    return X, conn, rng


def params(case):
    app = N.UNILATERAL if case.get("application") == "unilateral" else N.FULL
    if case["law"] == "elastic":
        dim = 2 if case.get("element") == "quad4" else 3
        return N.linear_elastic_params(dim, E0, NU, N.PLANE_STRAIN if case.get("plane") == "strain" else N.PLANE_STRESS)
    if case["law"] == "local":
        return N.local_damage_params(damage_application=app)
    return N.gradient_damage_params(
        damage_application=app, interaction=N.DECREASING if case.get("interaction") == "decreasing" else N.CONSTANT,
        interaction_r=DECREASING_R, interaction_eta=DECREASING_ETA)


def dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


def context(case, X, conn):
    """a Context with the mesh, the numbering and the pattern; the dof nodes' ranks and their number"""
    ct, dt, kind, order, nip = ELEMENTS[case["element"]]
    ranks, nn = N.dof_layer(ct, conn, dt)
    ctx = N.Context()
    ctx.set_cells(ct, X, conn)
    dim = X.shape[1]
    ctx.set_dof_type(0, dt, dim, dim * nn, N.cell_dofs(ranks, dim))
    if case["law"] == "gradient":
        ctx.set_dof_type(1, dt, 1, nn, N.cell_dofs(ranks, 1))
    ctx.set_integrand(params(case))
    ctx.set_rule(kind, order)
    ctx.build_pattern()
    return ctx, ranks, nn


def clamped(case, X, conn, ranks):
    """the dof nodes of the faces x = 0 and x = nx (corner nodes of the undistorted brick)"""
    corner = ranks[:, :conn.shape[1]].ravel()
    ix = conn.ravel() % (case["nx"] + 1)
    return np.unique(corner[ix == 0]), np.unique(corner[ix == case["nx"]])


# the load step: the face x = nx pulled to an average strain beyond kappa0 = f_t / E
LOAD_STRAIN = 1.1e-4


def prepare(case, seed):
    op = case["op"]
    if op in ("batch", "batch_adjoint"):
        return prepare_batch(case, seed)
    X, conn, rng = inputs(case, seed)
    ctx, ranks, nn = context(case, X, conn)
    nip = ELEMENTS[case["element"]][4]
    nc = len(conn)
    st = dict(op=op, ctx=ctx)
    if op == "load_step":
        theta = material_fields(rng, nc)
        ctx.set_material_fields(*theta)
        left, right = clamped(case, X, conn, ranks)
        eqs = [(int(3 * r + c), []) for r in left for c in range(3)] + [(int(3 * r), []) for r in right]
        ctx.set_constraints(0, eqs)
        rhs = np.zeros(len(eqs))
        rhs[3 * len(left):] = LOAD_STRAIN * case["nx"]
        st.update(rhs=dev(rhs), x=torch.zeros(ctx.n_rows, dtype=torch.float64, device="cuda"),
                  kappa=torch.zeros(nc * nip, dtype=torch.float64, device="cuda"))
        return st
    u, e, kappa = (dev(a) for a in state_arrays(rng, case["law"], X.shape[1], nn, nc * nip))
    if op == "solve":
        # f = K u for a u that satisfies the constraints
        left, _ = clamped(case, X, conn, ranks)
        ctx.set_constraints(0, [(int(3 * r + c), []) for r in left for c in range(3)])
        u.view(-1, 3)[torch.from_numpy(left).cuda().long()] = 0.0
        st.update(u=u, f=ctx.build_vector(u), K=torch.empty(ctx.nnz, dtype=torch.float64, device="cuda"),
                  x=torch.empty(ctx.n_rows, dtype=torch.float64, device="cuda"))
        return st
    st.update(u=u, e=e, kappa=kappa)
    if case.get("fields"):
        theta = material_fields(rng, nc)
        if op == "gradient":
            st.update(theta=dev(theta))
        else:
            ctx.set_material_fields(*theta)
    if op == "assemble":
        st.update(R=torch.empty(ctx.n_rows, dtype=torch.float64, device="cuda"),
                  K=torch.empty(ctx.nnz, dtype=torch.float64, device="cuda"))
    elif op == "gradient":
        st.update(r_obs=dev(rng.uniform(-1.0, 1.0, ctx.n_rows)))
    else:
        st.update(R=torch.empty(ctx.n_rows, dtype=torch.float64, device="cuda"),
                  stress=torch.empty(nc * nip * 6, dtype=torch.float64, device="cuda"))
    return st


def prepare_batch(case, seed):
    b = N.Batch()
    b.set_integrand(params(case))
    nc, nn_all = 0, 0
    for element, X, conn in batch_meshes(case, seed):
        ct, dt = ELEMENTS[element][:2]
        ranks, nn = N.dof_layer(ct, conn, dt)
        b.add_mesh(ct, dt, X, conn, ranks, nn)
        nc += len(conn)
        nn_all += nn
    sz = b.build()
    rng = np.random.default_rng([seed, 10**6])
    u, e, kappa = (dev(a) for a in state_arrays(rng, case["law"], 3, nn_all, sz["history"]))
    st = dict(op=case["op"], batch=b, u=u, e=e, kappa=kappa,
              R=torch.empty(sz["R"], dtype=torch.float64, device="cuda"),
              K=torch.empty(sz["K"], dtype=torch.float64, device="cuda"))
    if case["op"] == "batch":
        b.autotune(u, e, kappa, st["R"], st["K"])
    else:
        b.set_material_fields(*material_fields(rng, nc))
        st.update(r_obs=dev(rng.uniform(-1.0, 1.0, sz["R"])),
                  d_state=torch.empty(sz["R"], dtype=torch.float64, device="cuda"),
                  d_theta=torch.empty(sz["theta"], dtype=torch.float64, device="cuda"))
    return st


def run(st):
    op = st["op"]
    if op == "assemble":
        return st["ctx"].build_vector_matrix(st["u"], st["e"], st["kappa"], st["R"], st["K"])
    if op == "gradient":
        u, e, theta = (st[k].detach().requires_grad_() for k in ("u", "e", "theta"))
        R = N.autograd.residual(st["ctx"], u, e, st["kappa"], theta)
        return (R.detach(),) + torch.autograd.grad(R, (u, e, theta), R.detach() - st["r_obs"])
    if op == "explicit":
        ctx = st["ctx"]
        R = ctx.build_vector(st["u"], st["e"], st["kappa"], st["R"])
        kappa = ctx.update_history(st["u"], st["e"], st["kappa"])
        return R, kappa, ctx.eval_ip(N.IP_STRESS, st["u"], st["e"], kappa, st["stress"])
    if op == "batch":
        return st["batch"].assemble(st["u"], st["e"], st["kappa"], st["R"], st["K"])
    if op == "batch_adjoint":
        return st["batch"].residual_adjoint(st["u"], st["e"], st["kappa"], st["r_obs"], st["R"], st["K"], st["d_state"],
                                            st["d_theta"])
    if op == "solve":
        K = st["ctx"].build_matrix(st["u"], out=st["K"])
        return K, st["ctx"].solve(K, st["f"], method=N.SOLVER_CG, tol=1e-13, out=st["x"])[0]
    x, kappa = st["x"].clone(), st["kappa"].clone()
    st["ctx"].quasistatic_step(x, kappa, None, st["rhs"], tol=1e-9, max_iter=12, line_search_steps=0,
                              linear_tol=1e-12)
    return x, kappa


# ---- work ------------------------------------------------------------------------------------------------------------
def node_pairs(element, n):
    """ordered pairs of dof nodes that share a cell. The count is affine in each edge length: from the 8 smallest bricks"""
    def count(m):
        _, conn = brick_mesh(element, *m, 0.0, np.random.default_rng(0))
        ids = entity_ids(conn, EDGES[element], 10**4) if element in ("hex20", "tet10") else conn.astype(np.int64)
        keys, inv = np.unique(ids.ravel(), return_inverse=True)
        d = inv.reshape(ids.shape)
        nn = len(keys)
        pair = (d[:, :, None] * nn + d[:, None, :]).ravel()
        return len(np.unique(pair)), nn

    dims = 2 if element == "quad4" else 3
    c, d = np.zeros([2] * dims), np.zeros([2] * dims)
    for k in np.ndindex(*c.shape):
        c[k], d[k] = count(tuple(i + 1 for i in k) + (0,) * (3 - dims))
    out = []
    for f in (c, d):
        for i in range(dims):
            f = f[0] + (f[1] - f[0]) * (n[i] - 1)
        out.append(int(round(float(f))))
    return out


def mesh_work(element, law, n, matrix=True):
    """(cells, IPs, dof nodes, rows, nonzeros, bytes in, flops) of one mesh"""
    nip = ELEMENTS[element][4]
    dim = 2 if element == "quad4" else 3
    pairs, nn = node_pairs(element, n)
    nc = n[0] * n[1] * (n[2] if dim == 3 else 1) * (6 if element.startswith("tet") else 1)
    nnc = {"quad4": 4, "hex8": 8, "hex20": 8, "tet4": 4, "tet10": 4, "tet10iso": 10}[element]
    nnd = {"quad4": 4, "hex8": 8, "hex20": 20, "tet4": 4, "tet10": 10, "tet10iso": 10}[element]
    nodes_c = nn if element == "tet10iso" else (n[0] + 1) * (n[1] + 1) * (n[2] + 1)
    F = dim + (law == "gradient")
    byt = 8 * dim * nodes_c + 8 * F * nn + 4 * nc * (nnc + (nnd if nnd != nnc else 0)) + (0 if law == "elastic" else 8 * nc * nip)
    # per IP: Jacobian, gradients, strain, law and the residual; per node pair and IP the outer products of the tangent
    flops = nc * nip * (18 * nnc + 45 * nnd + 200)
    if matrix:
        flops += nc * nip * nnd * nnd * {"elastic": dim * dim * 2, "local": 36, "gradient": 50}[law]
    return dict(nc=nc, nip=nip, nn=nn, rows=F * nn, nnz=F * F * pairs, bytes=byt, flops=flops)


def work(case):
    op = case["op"]
    if op in ("batch", "batch_adjoint"):
        lay = np.random.default_rng(case["layout"])
        byt = flops = 0
        for _ in range(case["meshes"]):
            cells = np.exp(lay.uniform(np.log(case["lo"]), np.log(case["hi"])))
            element = ("tet4", "tet10", "hex8", "hex20")[lay.integers(4)] if op == "batch" else "hex8"
            bricks = cells / (6.0 if element.startswith("tet") else 1.0)
            n = max(1, round(bricks ** (1.0 / 3.0)))
            w = mesh_work(element, case["law"], (n, n, max(1, round(bricks / (n * n)))))
            byt += w["bytes"] + 8 * (w["rows"] + w["nnz"])
            flops += w["flops"]
            if op == "batch_adjoint":
                byt += 8 * (2 * w["rows"] + 6 * w["nc"])  # r_obs in, d_state out; fields in, d_theta out
                flops += w["nc"] * 8 * 1000
        return dict(bytes=byt, flops=flops)
    w = mesh_work(case["element"], case["law"], (case["nx"], case["ny"], case["nz"]), op not in ("gradient", "explicit"))
    byt, flops = w["bytes"], w["flops"]
    fields = 24 * w["nc"] if case.get("fields") else 0
    if op == "assemble":
        return dict(bytes=byt + fields + 8 * (w["rows"] + w["nnz"]), flops=flops)
    if op == "gradient":
        # forward: the inputs and R; backward: r_obs, the inputs again and the gradients
        return dict(bytes=byt + 2 * fields + 8 * 3 * w["rows"], flops=flops + w["nc"] * 8 * 1000)
    if op == "explicit":
        return dict(bytes=byt + 8 * (w["rows"] + w["nc"] * w["nip"] * 7), flops=flops)
    if op == "solve":
        # conjugate gradients: about 10 iterations per cell along an edge, each reading K and the vectors once
        its = 10 * max(case["nx"], case["ny"], case["nz"])
        return dict(bytes=byt + 8 * w["nnz"] + its * (8 * w["nnz"] + 80 * w["rows"]),
                    flops=flops + its * (2 * w["nnz"] + 14 * w["rows"]))
    # a load step: about 4 tangents and solves of 20 BiCGSTAB iterations per cell along the bar, two products each
    its = 4 * 20 * case["nx"]
    return dict(bytes=4 * (byt + 8 * w["nnz"]) + its * (16 * w["nnz"] + 160 * w["rows"]),
                flops=4 * flops + its * (4 * w["nnz"] + 30 * w["rows"]))


# ---- outputs from plain torch in 64 bits --------------------------------------------------------------------------------
def first_touch(ids):
    keys, first, inv = np.unique(ids.ravel(), return_index=True, return_inverse=True)
    rank = np.empty(len(keys), np.int64)
    rank[np.argsort(first)] = np.arange(len(keys))
    return rank[inv].reshape(ids.shape), len(keys)


def gauss(element):
    nip = ELEMENTS[element][4]
    if element.startswith("tet"):
        a, b = (5.0 - 5.0 ** 0.5) / 20.0, (5.0 + 3.0 * 5.0 ** 0.5) / 20.0
        xi = [[0.25] * 3] if nip == 1 else [[a, a, a], [b, a, a], [a, b, a], [a, a, b]]
        return np.array(xi), np.full(nip, 1.0 / (6.0 * nip))
    x, w = np.polynomial.legendre.leggauss(3 if nip == 27 else 2)
    dim = 2 if element == "quad4" else 3
    pts, wts = [], []
    for i in range(len(x) ** dim):
        k = [(i // len(x) ** d) % len(x) for d in range(dim)]
        pts.append([x[j] for j in k])
        wts.append(np.prod([w[j] for j in k]))
    return np.array(pts), np.array(wts)


HEX_NODES = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]], float)


def shape(kind, x):
    """shape functions at the point x (torch, differentiable)"""
    if kind == "quad4":
        s = torch.tensor(HEX_NODES[:4, :2])
        return ((1 + s[:, 0] * x[0]) * (1 + s[:, 1] * x[1])) / 4
    if kind in ("hex8", "hex20"):
        s = HEX_NODES
        if kind == "hex20":
            s = np.concatenate([s, np.array([0.5 * (s[a] + s[b]) for a, b in EDGES["hex20"]])])
        s = torch.tensor(s)
        f = torch.where(s == 0, 1 - x * x, 1 + s * x)
        p = f[:, 0] * f[:, 1] * f[:, 2]
        if kind == "hex8":
            return p / 8
        return torch.cat([p[:8] * ((s[:8] * x).sum(1) - 2) / 8, p[8:] / 4])
    L = torch.stack([1 - x.sum(), x[0], x[1], x[2]])
    if kind == "tet4":
        return L
    return torch.cat([L * (2 * L - 1), torch.stack([4 * L[a] * L[b] for a, b in EDGES["tet10"]])])


def shape_tables(kind, xi):
    pts = [torch.tensor(p) for p in xi]
    Nv = torch.stack([shape(kind, p) for p in pts])
    dN = torch.stack([torch.autograd.functional.jacobian(lambda y: shape(kind, y), p) for p in pts])
    return Nv, dN


class Reference:
    """One mesh (or one element type of a batch as one mesh): R, K and the integration-point fields of plain torch."""

    def __init__(self, case, element, X, conn, d, nn, theta, kappa):
        where = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: None if a is None else torch.as_tensor(a).to(where)  # noqa: E731
        ckind = {"hex20": "hex8", "tet10": "tet4", "tet10iso": "tet10"}.get(element, element)
        dkind = "tet10" if element == "tet10iso" else element
        xi, w = gauss(element)
        _, self.dNc = (t(a) for a in shape_tables(ckind, xi))
        self.Nd, self.dNd = (t(a) for a in shape_tables(dkind, xi))
        self.w, self.X, self.conn, self.d, self.nn = t(w), t(X), t(conn).long(), t(d).long(), nn
        self.case, self.element, self.dim = case, element, X.shape[1]
        self.nip, self.nc = len(w), len(conn)
        self.theta, self.kappa = t(theta), None if kappa is None else t(kappa).view(self.nip, self.nc).T
        self.two = case["law"] == "gradient"
        self.where = where

    def chunks(self):
        n = max(1, 40_000_000 // (self.nip * self.d.shape[1] * 20))
        return [slice(i, min(i + n, self.nc)) for i in range(0, self.nc, n)]

    def geometry(self, c):
        J = torch.einsum("cni,qnk->cqik", self.X[self.conn[c]], self.dNc)
        inv = torch.linalg.inv(J)
        return torch.einsum("qnl,cqlk->cqnk", self.dNd, inv), torch.linalg.det(J) * self.w

    def points(self, c, g, ue, ee, theta=None):
        """stress, kappa, damage and equivalent strain, nonlocal strain at the integration points"""
        H = torch.einsum("cni,cqnk->cqik", ue, g)
        eps = 0.5 * (H + H.transpose(2, 3))
        eye = torch.eye(self.dim, dtype=torch.float64, device=eps.device)
        tr = eps.diagonal(dim1=2, dim2=3).sum(2)[..., None, None]
        if self.case["law"] == "elastic":
            lam, mu = E0 * NU / ((1 + NU) * (1 - 2 * NU)), E0 / (2 * (1 + NU))
            if self.dim == 2 and self.case.get("plane") != "strain":
                lam = 2 * lam * mu / (lam + 2 * mu)
            return lam * tr * eye + 2 * mu * eps, None, None, None, None
        E, k0, beta = E0, KAPPA0, BETA
        if theta is None and self.theta is not None:
            theta = self.theta[:, c]
        if theta is not None:
            E, k0, beta = theta[0][:, None], (theta[1] / theta[0])[:, None], (theta[1] / theta[2])[:, None]
        I1 = tr[..., 0, 0]
        dv = eps - tr * eye / 3
        J2 = 0.5 * (dv * dv).sum((2, 3))
        K1 = (MISES_K - 1) / (2 * MISES_K * (1 - 2 * NU))
        K2 = 3 / (MISES_K * (1 + NU) ** 2)
        q2 = K1 * K1 * I1 * I1 + K2 * J2
        eq = K1 * I1 + torch.where(q2 > 0, torch.sqrt(torch.where(q2 > 0, q2, 1.0)), 0.0)  # derivative 0 at 0
        eN = torch.einsum("qn,cn->cq", self.Nd, ee) if self.two else None
        kap = torch.maximum(self.kappa[c], eN if self.two else eq)
        r = k0 / torch.where(kap < k0, torch.ones_like(kap), kap)
        om = torch.where(kap < k0, torch.zeros_like(kap), 1 - r * (1 - ALPHA + ALPHA * torch.exp(beta * (k0 - kap))))
        on = torch.where(I1 < 0, 0.0, 1.0).double() if self.case.get("application") == "unilateral" else 1.0
        k3, g2 = 3 * E / (3 - 6 * NU), 2 * E / (2 + 2 * NU)
        sig = ((1 - om * on) * k3 * I1 / 3)[..., None, None] * eye + ((1 - om) * g2)[..., None, None] * dv
        return sig, kap, om, eq, eN

    def cell_residual(self, c, g, s, ue, ee, theta=None):
        sig, _, om, eq, eN = self.points(c, g, ue, ee, theta)
        ru = torch.einsum("cq,cqnk,cqik->cni", s, g, sig)
        if not self.two:
            return ru
        ge = torch.einsum("cn,cqnk->cqk", ee, g)
        f = 1.0
        if self.case.get("interaction") == "decreasing":
            z = float(np.exp(-DECREASING_ETA))
            f = (((1 - DECREASING_R) * torch.exp(-DECREASING_ETA * om) + DECREASING_R - z) / (1 - z))[..., None]
        re = torch.einsum("cq,qn->cn", s * (eN - eq), self.Nd) + NONLOCAL_C * torch.einsum("cq,cqnk,cqk->cn", s, g, f * ge)
        return torch.cat([ru, re[..., None]], 2)

    def cell_state(self, c, x):
        u = x[:self.dim * self.nn].view(-1, self.dim)[self.d[c]]
        return u, x[self.dim * self.nn:][self.d[c]] if self.two else None

    def vector(self, x, theta=None):
        F = self.dim + self.two
        out = torch.zeros(self.nn, F, dtype=torch.float64, device=self.where)
        for c in self.chunks():
            g, s = self.geometry(c)
            r = self.cell_residual(c, g, s, *self.cell_state(c, x), None if theta is None else theta[:, c])
            out = out.index_add(0, self.d[c].reshape(-1), r.reshape(-1, F))
        return torch.cat([out[:, :self.dim].reshape(-1), out[:, self.dim:].reshape(-1)])

    def cell_matrices(self, c, x):
        """K_e columns by forward differentiation of the residual: yields (column node b, component, rows (cells, n, F))"""
        g, s = self.geometry(c)
        ue, ee = self.cell_state(c, x)
        F = self.dim + self.two
        for b in range(self.d.shape[1]):
            for k in range(F):
                du = torch.zeros_like(ue)
                de = torch.zeros_like(ee) if self.two else None
                if k < self.dim:
                    du[:, b, k] = 1.0
                else:
                    de[:, b] = 1.0
                if self.two:
                    _, col = torch.func.jvp(lambda p, q: self.cell_residual(c, g, s, p, q), (ue, ee), (du, de))
                else:
                    _, col = torch.func.jvp(lambda p: self.cell_residual(c, g, s, p, None), (ue,), (du,))
                yield b, k, col

    def matrix(self, x):
        """values of the CSR: rows [u; e], columns [u, e] ascending"""
        F, nn, n = self.dim + self.two, self.nn, self.d.shape[1]
        keys = (self.d[:, :, None] * nn + self.d[:, None, :]).reshape(-1)
        uniq, inv = torch.unique(keys, return_inverse=True)
        del keys
        inv = inv.view(self.nc, n, n)
        nadj = torch.bincount(uniq // nn, minlength=nn)
        ptr = torch.cumsum(nadj, 0) - nadj
        K = torch.zeros(F * F * len(uniq), dtype=torch.float64, device=self.where)
        comp = torch.arange(F, device=self.where)
        base_e = F * self.dim * len(uniq)
        for c in self.chunks():
            a = self.d[c]
            first = torch.where(comp < self.dim, F * (self.dim * ptr[a][..., None] + comp * nadj[a][..., None]),
                                base_e + F * ptr[a][..., None])
            for b, k, col in self.cell_matrices(c, x):
                slot = inv[c, :, b] - ptr[a]
                at = slot * self.dim + k if k < self.dim else self.dim * nadj[a] + slot
                K.index_add_(0, (first + at[..., None]).reshape(-1), col.reshape(-1))
        return K


def exact_mesh(case, seed):
    X, conn, rng = inputs(case, seed)
    element = case["element"]
    ids = entity_ids(conn, EDGES[element], len(X)) if element in ("hex20", "tet10") else conn.astype(np.int64)
    d, nn = first_touch(ids)
    return X, conn, rng, d, nn


def exact(case, seed):
    if case["op"] in ("batch", "batch_adjoint"):
        return exact_batch(case, seed)
    X, conn, rng, d, nn = exact_mesh(case, seed)
    op, nip, nc = case["op"], ELEMENTS[case["element"]][4], len(conn)
    if op == "load_step":
        return exact_load_step(case, X, conn, d, nn, material_fields(rng, nc))
    u, e, kappa = state_arrays(rng, case["law"], X.shape[1], nn, nc * nip)
    if op == "solve":
        left, _ = clamped(case, X, conn, d)
        u.reshape(-1, 3)[left] = 0.0
        ref = Reference(case, case["element"], X, conn, d, nn, None, None)
        u = torch.from_numpy(u).to(ref.where)
        return ref.matrix(u), u
    theta = material_fields(rng, nc) if case.get("fields") else None
    ref = Reference(case, case["element"], X, conn, d, nn, theta, kappa)
    x = torch.from_numpy(u if e is None else np.concatenate([u, e])).to(ref.where)
    if op == "assemble":
        return ref.vector(x), ref.matrix(x)
    if op == "gradient":
        r_obs = torch.from_numpy(rng.uniform(-1.0, 1.0, len(x))).to(ref.where)
        R = ref.vector(x)
        gx, gt = vector_gradient(ref, x, ref.theta, R - r_obs)
        return R, gx[:3 * nn], gx[3 * nn:], gt
    R = ref.vector(x)
    stress = torch.empty(nc, nip, 6, dtype=torch.float64, device=ref.where)
    hist = torch.empty_like(ref.kappa)
    for c in ref.chunks():
        g, _ = ref.geometry(c)
        sig, kap, *_ = ref.points(c, g, *ref.cell_state(c, x))
        stress[c] = torch.stack([sig[..., i, j] for i, j in ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))], -1)
        hist[c] = kap
    return R, hist.T.reshape(-1), stress


def vector_gradient(ref, x, theta, lam):
    """(dR/dx)^T lam and (dR/dtheta)^T lam, cell chunk by cell chunk"""
    gx, gt = torch.zeros_like(x), torch.zeros_like(theta)
    nu = ref.dim * ref.nn
    for c in ref.chunks():
        g, s = ref.geometry(c)
        ue, ee = (v.detach().requires_grad_() for v in ref.cell_state(c, x))
        th = theta[:, c].detach().requires_grad_()
        lu, le = ref.cell_state(c, lam)
        r = ref.cell_residual(c, g, s, ue, ee, th)
        du, de, dt = torch.autograd.grad((r * torch.cat([lu, le[..., None]], 2)).sum(), (ue, ee, th))
        gx[:nu].view(-1, ref.dim).index_add_(0, ref.d[c].reshape(-1), du.reshape(-1, ref.dim))
        gx[nu:].index_add_(0, ref.d[c].reshape(-1), de.reshape(-1))
        gt[:, c] = dt
    return gx, gt


def exact_load_step(case, X, conn, d, nn, theta):
    """Newton with dense direct solves from the unloaded state to the converged one"""
    nc = len(conn)
    ref = Reference(case, case["element"], X, conn, d, nn, theta, np.zeros(nc * 8))
    left, right = (torch.from_numpy(v).to(ref.where) for v in clamped(case, X, conn, d))
    n = 4 * nn
    free = torch.ones(n, dtype=torch.bool, device=ref.where)
    for c in range(3):
        free[3 * left + c] = False
    free[3 * right] = False
    step = torch.zeros(n, dtype=torch.float64, device=ref.where)
    step[3 * right] = LOAD_STRAIN * case["nx"]
    x = torch.zeros_like(step)
    rows = torch.cat([3 * ref.d[..., None] + torch.arange(3, device=ref.where), 3 * nn + ref.d[..., None]], 2).reshape(nc, -1)
    last = float("inf")
    for it in range(30):
        K = torch.zeros(n, n, dtype=torch.float64, device=ref.where)
        for c in ref.chunks():
            for b, k, col in ref.cell_matrices(c, x):
                j = rows[c, 4 * b + k]
                K.view(-1).index_add_(0, (rows[c] * n + j[:, None]).reshape(-1), col.reshape(len(j), -1).reshape(-1))
        move = step if it == 0 else torch.zeros_like(step)
        r = ref.vector(x) + K @ move
        dx = torch.zeros_like(x)
        dx[free] = torch.linalg.solve(K[free][:, free], r[free])
        x = x + move - dx
        now = float(torch.linalg.vector_norm(dx) / torch.linalg.vector_norm(x))
        if it > 0 and now < 1e-13 or it > 3 and now > 0.5 * last and now < 1e-11:
            break
        last = now
    kap = torch.einsum("qn,cn->cq", ref.Nd, x[3 * nn:][ref.d])
    return x, torch.maximum(kap, torch.zeros_like(kap)).T.reshape(-1)


def exact_batch(case, seed):
    meshes = batch_meshes(case, seed)
    rng = np.random.default_rng([seed, 10**6])
    parts, base = [], 0
    for element, X, conn in meshes:
        ids = entity_ids(conn, EDGES[element], len(X)) if element in ("hex20", "tet10") else conn.astype(np.int64)
        parts.append((element, X, conn, *first_touch(ids), base))
        base += len(conn)
    nn_all = sum(p[4] for p in parts)
    n_hist = sum(len(p[2]) * ELEMENTS[p[0]][4] for p in parts)
    u, e, kappa = state_arrays(rng, case["law"], 3, nn_all, n_hist)
    adjoint = case["op"] == "batch_adjoint"
    theta = material_fields(rng, base) if adjoint else None
    r_obs = rng.uniform(-1.0, 1.0, 4 * nn_all) if adjoint else None
    out = [[], [], [], []]
    nodes = hist = row = 0
    for element in BATCH_ORDER:
        group = [p for p in parts if p[0] == element]
        if not group:
            continue
        X = np.concatenate([p[1] for p in group])
        xo = np.cumsum([0] + [len(p[1]) for p in group])
        no = np.cumsum([0] + [p[4] for p in group])
        conn = np.concatenate([p[2].astype(np.int64) + o for p, o in zip(group, xo)])
        d = np.concatenate([p[3] + o for p, o in zip(group, no)])
        nn, nh = int(no[-1]), len(conn) * ELEMENTS[element][4]
        th = None if theta is None else np.concatenate([theta[:, p[5]:p[5] + len(p[2])] for p in group], 1)
        ref = Reference(case, element, X, conn, d, nn, th, None if kappa is None else kappa[hist:hist + nh])
        xs = u[3 * nodes:3 * (nodes + nn)]
        x = torch.from_numpy(xs if e is None else np.concatenate([xs, e[nodes:nodes + nn]])).to(ref.where)
        out[0].append(ref.vector(x))
        out[1].append(ref.matrix(x))
        if adjoint:
            lam = out[0][-1] - torch.from_numpy(r_obs[row:row + len(x)]).to(ref.where)
            gx, gt = vector_gradient(ref, x, ref.theta, lam)
            out[2].append(gx)
            out[3].append(gt.reshape(-1))
        nodes, hist, row = nodes + nn, hist + nh, row + len(x)
    return tuple(torch.cat(v) for v in out if v)
