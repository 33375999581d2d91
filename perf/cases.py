"""Performance cases of the element -> assembly -> solve path, from the smallest call to the largest.

A case is a dict of plain values whose ``task`` names the entry point:

* ``analysis``  -- ``FiniteElementAnalysis`` built from node loads and conditions, then ``solve()``: the
  drop-in call of a script that has one plane problem.  Host lowering, pattern, upload and a short PCG.
* ``solve``     -- the array-level solve of a program that keeps the mesh and changes the materials:
  assembly, elimination, preconditioner set-up and PCG (``FESystem`` and ``solve_reduced``).
* ``batch``     -- many independent uneven plates in one call (``MeshBatch.solve``).
* ``assemble``  -- the assembled stiffness or mass matrix in one of its layouts.
* ``fields``    -- strain, stress and energy (or B) of every element after a solve.
* ``modal``     -- the lowest modes of several stiffness draws of one mesh (``modal.lobpcg``).
* ``train``     -- loss and gradient of the learned preconditioner on one system (forward and backward).

Meshes are the structured ones of ``meshgen`` (``numbering='shuffled'`` renumbers the nodes at random, as
an unstructured mesh generator's numbering looks to the memory system).  The mesh, its pattern and the
coarse space are what a program keeps from one call to the next; materials, loads and start vectors come
from the seed.
"""

import copy
import functools
import math
import os

import numpy as np
import torch

from finite_elements_amd import _hip, analysis, conditions, device, learned, loads, meshgen, modal
from finite_elements_amd.batch import MeshBatch
from finite_elements_amd.mesh import ArrayMesh
from finite_elements_amd.system import FESystem

LAYOUTS = {'planes': _hip.FE_LAYOUT_PLANES, 'bsr': _hip.FE_LAYOUT_BSR, 'csr': _hip.FE_LAYOUT_CSR}
PLANE_STRESS = 2


def listed():
    return [
        # one small plane-stress cantilever through the drop-in class: launch and host latency
        {'name': 'analysis_40x10', 'task': 'analysis', 'nx': 40, 'ny': 10, 'precond': 'block_jacobi',
         'precision': 'fp64'},
        # a small 3D part with solve()'s defaults (FP64, Jacobi)
        {'name': 'solve_cube13_jacobi', 'task': 'solve', 'problem': 'cube', 'n': 13, 'numbering': 'grid',
         'precond': 'jacobi', 'precision': 'fp64'},
        # an ordinary 3D part whose nodes are numbered as a mesh generator leaves them
        {'name': 'solve_cube27_shuffled', 'task': 'solve', 'problem': 'cube', 'n': 27,
         'numbering': 'shuffled', 'precond': 'two_level', 'precision': 'mixed'},
        # a plane magnetostatics of ordinary size, all in FP64
        {'name': 'solve_magnetic150_fp64', 'task': 'solve', 'problem': 'magnetic', 'n': 150,
         'numbering': 'grid', 'precond': 'block_jacobi', 'precision': 'fp64'},
        # the large magnetostatics with the recommended method
        {'name': 'solve_magnetic450', 'task': 'solve', 'problem': 'magnetic', 'n': 450, 'numbering': 'grid',
         'precond': 'two_level', 'precision': 'mixed'},
        # the largest single system: 64^3 cells, lognormal stiffness
        {'name': 'solve_cube64', 'task': 'solve', 'problem': 'cube', 'n': 64, 'numbering': 'grid',
         'precond': 'two_level', 'precision': 'mixed'},
        # a design study: uneven plates in one batch
        {'name': 'batch_256', 'task': 'batch', 'count': 256, 'geometry': 3, 'precond': 'two_level',
         'precision': 'fp64'},
        # stiffness of the large cube in the solver's layout
        {'name': 'assemble_cube64', 'task': 'assemble', 'problem': 'cube', 'n': 64, 'numbering': 'grid',
         'what': 'stiffness', 'layout': 'planes'},
        # consistent mass of a plate as scalar CSR (what m_matrix hands to scipy)
        {'name': 'assemble_plate_mass_csr', 'task': 'assemble', 'problem': 'plate', 'n': 301,
         'numbering': 'grid', 'what': 'mass', 'layout': 'csr'},
        # post-processing of a 3D solution
        {'name': 'fields_cube48', 'task': 'fields', 'problem': 'cube', 'n': 48, 'numbering': 'grid'},
        # a modal study: stiffness draws of one part
        {'name': 'modal_20_8', 'task': 'modal', 'n': 20, 'variants': 8, 'modes': 8},
        # one training system of the learned preconditioner
        {'name': 'train_cube24', 'task': 'train', 'n': 24},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def precision(precond):
        # FP32 iterations go with the preconditioner that keeps them few; the others run in FP64
        return rng.choice(['fp64', 'mixed', 'mixed']) if precond == 'two_level' else 'fp64'

    task = rng.choice(['analysis', 'solve', 'solve', 'solve', 'solve', 'batch', 'assemble', 'assemble',
                       'fields', 'modal', 'train'])
    numbering = rng.choice(['grid', 'grid', 'shuffled'])
    if task == 'analysis':
        precond = rng.choice(['jacobi', 'block_jacobi', 'two_level'])
        return {'task': task, 'nx': log_int(12, 120), 'ny': log_int(4, 40), 'precond': precond,
                'precision': precision(precond)}
    if task == 'solve':
        problem = rng.choice(['cube', 'cube', 'magnetic', 'plate'])
        precond = rng.choice(['jacobi', 'block_jacobi', 'two_level', 'two_level'])
        # a large system is not solved without the coarse correction
        largest = {'cube': (40, 60), 'magnetic': (250, 449), 'plate': (100, 160)}[problem]
        n = log_int({'cube': 6, 'magnetic': 40, 'plate': 16}[problem], largest[precond == 'two_level'])
        return {'task': task, 'problem': problem, 'n': n, 'numbering': numbering, 'precond': precond,
                'precision': precision(precond)}
    if task == 'batch':
        precond = rng.choice(['block_jacobi', 'two_level', 'two_level'])
        return {'task': task, 'count': log_int(2, 256), 'geometry': rng.randrange(1000),
                'precond': precond, 'precision': precision(precond)}
    if task == 'modal':
        return {'task': task, 'n': rng.randrange(6, 19), 'variants': rng.randrange(1, 9),
                'modes': rng.randrange(3, 8)}
    if task == 'train':
        return {'task': task, 'n': log_int(6, 23)}
    problem = rng.choice(['cube', 'plate', 'magnetic'])
    if task == 'fields':
        return {'task': task, 'problem': problem, 'numbering': numbering,
                'n': log_int(6, 47) if problem == 'cube' else log_int(20, 640)}
    n = log_int(6, 63) if problem == 'cube' else log_int(20, 640)
    return {'task': task, 'problem': problem, 'n': n, 'numbering': numbering,
            'what': 'stiffness' if problem == 'magnetic' else rng.choice(['stiffness', 'mass']),
            'layout': rng.choice(['planes', 'bsr', 'csr'])}


# ------------------------------------------------------------------------------------------------
# problems: the mesh and constraints of a case, and the materials and loads of a seed
# ------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=24)
def _mesh(problem, n, numbering):
    """(kind, coords, conn, fixed DOFs) of a case; nothing here depends on a seed."""
    if problem == 'cube':
        kind, (coords, conn) = 'tet_elastic', meshgen.kuhn_tets(n)
    elif problem == 'plate':
        kind, (coords, conn) = 'tri_elastic', meshgen.structured_tri(n, max(1, n // 2), 1.0, 0.5)
    else:
        kind, (coords, conn) = 'tri_magnetic', meshgen.structured_tri(n, n, 2.0, 2.0, -1.0, -1.0)
    if numbering == 'shuffled':
        new = np.random.default_rng(n).permutation(coords.shape[0])
        old = np.argsort(new)
        coords, conn = coords[old], new[conn].astype(np.int32)
    d = {'cube': 3, 'plate': 2, 'magnetic': 1}[problem]
    if problem == 'cube':
        held = np.flatnonzero(coords[:, 2] == 0.0)
    elif problem == 'plate':
        held = np.flatnonzero(coords[:, 0] == 0.0)
    else:
        held = np.flatnonzero(np.abs(coords).max(axis=1) >= 1.0)
    fixed = (held[:, None] * d + np.arange(d)[None, :]).ravel()
    return kind, np.ascontiguousarray(coords), np.ascontiguousarray(conn), fixed


def _materials(problem, n, coords, conn, seed):
    rng = np.random.default_rng(seed)
    ne = conn.shape[0]
    if problem == 'cube':  # lognormal field with a correlation length of a tenth of the edge
        side = 2 * n
        white = np.fft.rfftn(rng.standard_normal((side, side, side)).astype(np.float32))
        k = 2 * np.pi * n * np.fft.fftfreq(side)
        kr = 2 * np.pi * n * np.fft.rfftfreq(side)
        decay = [np.exp(-0.25 * 0.01 * q ** 2) for q in (k, k, kr)]
        white *= decay[0][:, None, None] * decay[1][None, :, None] * decay[2][None, None, :]
        field = np.fft.irfftn(white, s=(side, side, side), axes=(0, 1, 2))[:n, :n, :n]
        field = (field - field.mean()) / field.std()
        E = np.repeat(1e11 * np.exp(field.ravel().astype(np.float64) - 0.5), 6)
        return {'E': E, 'nu': np.full(ne, 0.3), 'rho': rng.uniform(7000.0, 8000.0, ne)}
    if problem == 'plate':
        return {'E': 1.4e11 * np.exp(0.5 * rng.standard_normal(ne)), 'nu': rng.uniform(0.25, 0.35, ne),
                'thickness': np.full(ne, 0.01), 'rho': rng.uniform(7000.0, 8000.0, ne)}
    r = np.hypot(*coords[conn].mean(axis=1).T)
    iron = rng.uniform(500.0, 1500.0)
    return {'mu': meshgen.MU0 * np.where((r >= 0.3) & (r <= 0.45), iron, 1.0)}


def _load(problem, coords, seed):
    """Nodal loads: tractions on the face opposite the clamp, or two coils of opposite current."""
    rng = np.random.default_rng(seed + 1)
    if problem == 'magnetic':
        x, y = coords.T
        J = rng.uniform(0.5e6, 1.5e6)
        inside = (np.abs(y) <= 0.1) & (np.abs(x) >= 0.15) & (np.abs(x) <= 0.25)
        return J * 4.0 / coords.shape[0] * np.where(inside, np.where(x < 0, 1.0, -1.0), 0.0)
    axis = 2 if problem == 'cube' else 0
    d = coords.shape[1]
    far = np.flatnonzero(coords[:, axis] == coords[:, axis].max())
    f = np.zeros((coords.shape[0], d))
    f[far] = rng.uniform(-1e6, 1e6, d)[None, :] / far.size
    return f.ravel()


@functools.lru_cache(maxsize=24)
def _system(problem, n, numbering):
    """The device system of a mesh: pattern, graph and schedules, kept by a program that solves on it
    again with other materials."""
    kind, coords, conn, fixed = _mesh(problem, n, numbering)
    return FESystem(kind, coords, conn, _materials(problem, n, coords, conn, 0),
                    plane_mode=PLANE_STRESS if problem == 'plate' else 0)


def _seeded_system(case, seed):
    problem, n, numbering = case['problem'], case['n'], case['numbering']
    kind, coords, conn, fixed = _mesh(problem, n, numbering)
    base = _system(problem, n, numbering)
    if case.get('precond') == 'two_level':
        base.coarse_space(fixed)  # once per mesh; the copies below share it
    sysm = copy.copy(base)
    sysm.set_materials(_materials(problem, n, coords, conn, seed))
    return sysm, coords, fixed


def _plate_problem(nx, ny, rng):
    """One plane-stress plate of a design study, 1 cm cells: x = 0 clamped, a unit tip load."""
    h = 0.01
    coords, conn = meshgen.structured_tri(nx, ny, nx * h, ny * h)
    ne = conn.shape[0]
    mats = {'E': 1.4e11 * np.exp(0.5 * rng.standard_normal(ne)), 'nu': rng.uniform(0.25, 0.35, ne),
            'thickness': np.full(ne, 0.01), 'rho': np.full(ne, 7850.0)}
    left = np.flatnonzero(coords[:, 0] == 0.0)
    fixed = np.sort(np.concatenate([2 * left, 2 * left + 1]))
    theta = rng.uniform(0, 2 * np.pi)
    tip = (ny // 2) * (nx + 1) + nx
    f = np.zeros(coords.shape[0] * 2)
    f[2 * tip], f[2 * tip + 1] = math.cos(theta), math.sin(theta)
    return meshgen.Problem('plate', 'tri_elastic', coords, conn, mats, plane_mode=PLANE_STRESS,
                           fixed_dofs=fixed, fixed_values=np.zeros(fixed.size), f=f)


def _plate_sizes(case):
    rng = np.random.default_rng(case['geometry'])
    return [(int(rng.integers(20, 97)), int(rng.integers(10, 41))) for _ in range(case['count'])]


def _plate_problems(case, seed):
    rng = np.random.default_rng(seed)
    return [_plate_problem(nx, ny, rng) for nx, ny in _plate_sizes(case)]


@functools.lru_cache(maxsize=4)
def _batch(count, geometry):
    mb = MeshBatch(_plate_problems({'count': count, 'geometry': geometry}, 0))
    mb.coarse_space()
    return mb


#: relative residual of the solves and eigenpairs: a program that wants nine digits of the result
TOL = 1e-10


# ------------------------------------------------------------------------------------------------
# prepare and run
# ------------------------------------------------------------------------------------------------
def prepare(case, seed):
    task = case['task']
    st = {'task': task, 'case': case}
    if task == 'analysis':
        nx, ny = case['nx'], case['ny']
        pr = meshgen.cantilever_2d(nx, ny, lx=0.025 * nx, ly=0.025 * ny)
        rng = np.random.default_rng(seed)
        pr.materials['E'] = 210e9 * np.exp(0.2 * rng.standard_normal(pr.conn.shape[0]))
        am = ArrayMesh(pr.coords, pr.conn, pr.kind, pr.materials)
        nodes, tip = am.nodes, pr.meta['tip_node']
        st['mesh'] = am
        st['loads'] = [loads.NodeLoad(nodes[tip], float(v), k + 1)
                       for k, v in enumerate(rng.uniform(-1e4, 1e4, 2))]
        st['bcs'] = [conditions.NodeBoundaryCondition(nodes[q // 2], 0.0, int(q % 2) + 1)
                     for q in pr.fixed_dofs]
        return st
    if task == 'batch':
        base = _batch(case['count'], case['geometry'])
        problems = _plate_problems(case, seed)
        mb = copy.copy(base)
        mb.problems = problems
        mb.sysm = copy.copy(base.sysm)
        mb.sysm.set_materials({k: np.concatenate([p.materials[k] for p in problems])
                               for k in problems[0].materials})
        mb.f = np.concatenate([p.f for p in problems])
        mb._fixed = None
        st['batch'] = mb
        return st
    if task == 'modal':
        kind, coords, conn, fixed = _mesh('cube', case['n'], 'grid')
        base = _system('cube', case['n'], 'grid')
        st['fixed'], _ = base.dirichlet(fixed)
        st['coarse'] = base.coarse_space(fixed)
        st['mass'] = device.apply_dirichlet(base.mass_bsr(), st['fixed'])
        st['systems'] = []
        for E in _modal_moduli(case, seed):
            s = copy.copy(base)
            s.set_materials({'E': E, 'nu': np.full(E.size, 0.3), 'rho': np.full(E.size, 7850.0)})
            st['systems'].append(s)
        st['seed'] = seed
        rng = np.random.default_rng(seed + 4)
        st['reference'] = base.ctx.tensor(rng.standard_normal(coords.size))
        return st
    if task == 'train':
        full = {'problem': 'cube', 'n': case['n'], 'numbering': 'grid'}
        sysm, coords, fixed = _seeded_system(full, seed)
        mask, g = sysm.dirichlet(fixed)
        KD, _ = sysm.prepare(sysm.stiffness_bsr(), mask, g, torch.zeros_like(g))
        pairs = []
        for e in _train_errors(coords, fixed, seed):
            e = sysm.ctx.tensor(e)
            pairs.append((device.spmv(KD, e), e))
        st['model'] = learned.LearnedPreconditioner.load(_WEIGHTS)
        st['sample'] = learned.TrainingSystem(KD, mask, pairs, device.precond_setup(KD, 'block_jacobi'))
        st['grad'] = torch.zeros_like(st['model'].params(sysm.ctx))
        return st
    sysm, coords, fixed = _seeded_system(case, seed)
    st['sysm'] = sysm
    if task == 'solve':
        st['fixed'], st['g'] = sysm.dirichlet(fixed)
        st['f'] = sysm.ctx.tensor(_load(case['problem'], coords, seed))
        st['coarse'] = sysm.coarse_space(fixed) if case['precond'] == 'two_level' else None
    elif task == 'fields':
        st['u'] = sysm.ctx.tensor(_displacement(case['problem'], coords, seed))
    return st


def run(st):
    case, task = st['case'], st['task']
    if task == 'analysis':
        an = analysis.FiniteElementAnalysis(st['mesh'], [], [], st['loads'], [], [], st['bcs'], [], [],
                                            plane_strain=False, plane_stress=True)
        res = an.solve(tol=TOL, precond=case['precond'], precision=case['precision'])
        return np.asarray(res.result_vector)
    if task == 'solve':
        sysm = st['sysm']
        K = sysm.stiffness_bsr()
        KD, b = sysm.prepare(K, st['fixed'], st['g'], st['f'], coarse=st['coarse'])
        u, _ = analysis.solve_reduced(sysm, KD, b, st['fixed'], case['precond'], case['precision'],
                                      tol=TOL, coarse=st['coarse'])
        return u
    if task == 'batch':
        u, _ = st['batch'].solve(tol=TOL, precision=case['precision'], precond=case['precond'])
        return u
    if task == 'assemble':
        sysm, layout = st['sysm'], LAYOUTS[case['layout']]
        return sysm.stiffness(layout) if case['what'] == 'stiffness' else sysm.mass(layout)
    if task == 'fields':
        return st['sysm'].element_fields(st['u'])
    if task == 'modal':
        KDs = [device.apply_dirichlet(s.stiffness_bsr(), st['fixed']) for s in st['systems']]
        vals, vecs, _ = modal.lobpcg(KDs, st['mass'], case['modes'], fixed=st['fixed'], tol=TOL,
                                     coarse=st['coarse'], streams=min(2, len(KDs)), seed=st['seed'])
        # a shape's sign is the program's choice: a positive product with its reference vector
        return {'vals': vals, 'vecs': vecs * torch.sign(st['reference'] @ vecs)[:, None, :]}
    st['grad'].zero_()
    return {'loss': st['model'].loss_and_grad(st['sample'], st['grad']), 'grad': st['grad']}


_WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(learned.__file__)), 'weights',
                        'learned_block_jacobi_tet.npz')


def _modal_moduli(case, seed):
    rng = np.random.default_rng(seed)
    return [210e9 * np.exp(math.log(1.2) * rng.standard_normal(6 * case['n'] ** 3))
            for _ in range(case['variants'])]


def _train_errors(coords, fixed, seed):
    """A rough and a smooth error vector, zero at the clamp."""
    rng = np.random.default_rng(seed + 2)
    rough = rng.standard_normal(coords.shape[0] * 3)
    k = rng.uniform(1.0, 4.0, (3, 3))
    smooth = np.sin(coords @ k).ravel()
    for e in (rough, smooth):
        e[fixed] = 0.0
    return rough, smooth


def _displacement(problem, coords, seed):
    """A smooth field of solution-like size with a little roughness."""
    rng = np.random.default_rng(seed + 3)
    d = {'cube': 3, 'plate': 2, 'magnetic': 1}[problem]
    k = rng.uniform(0.5, 3.0, (coords.shape[1], d))
    return (1e-3 * np.sin(coords @ k) + 1e-6 * rng.standard_normal((coords.shape[0], d))).ravel()


# ------------------------------------------------------------------------------------------------
# work: inputs read once, outputs written once; operations of one evaluation of what is computed
# ------------------------------------------------------------------------------------------------
def _counts(problem, n):
    """(nodes, elements, node blocks of the matrix) of a structured mesh."""
    if problem == 'cube':
        m = n + 1
        return m ** 3, 6 * n ** 3, m ** 3 + 2 * (3 * n * m * m + 3 * n * n * m + n ** 3)
    nx, ny = (n, n) if problem == 'magnetic' else (n, max(1, n // 2))
    return ((nx + 1) * (ny + 1), 2 * nx * ny,
            (nx + 1) * (ny + 1) + 2 * (nx * (ny + 1) + ny * (nx + 1) + nx * ny))


def _mesh_bytes(problem, n):
    nodes, elems, _ = _counts(problem, n)
    dim, npe, mats = {'cube': (3, 4, 2), 'plate': (2, 3, 3), 'magnetic': (2, 3, 1)}[problem]
    return 8 * dim * nodes + (4 * npe + 8 * mats) * elems


def _solve_work(problem, n):
    """One assembly, and one application of the matrix (a solver cannot do with less)."""
    d = {'cube': 3, 'plate': 2, 'magnetic': 1}[problem]
    nodes, elems, blocks = _counts(problem, n)
    npe = 4 if problem == 'cube' else 3
    return {'bytes': _mesh_bytes(problem, n) + (8 * d * d + 4) * blocks + 3 * 8 * d * nodes,
            'flops': 6 * (npe * d) ** 2 * elems + 2 * d * d * blocks}


def work(case):
    task = case['task']
    if task == 'analysis':
        nodes, elems = (case['nx'] + 1) * (case['ny'] + 1), 2 * case['nx'] * case['ny']
        return {'bytes': 36 * elems + 16 * nodes + 7 * 36 * nodes + 48 * nodes, 'flops': 216 * elems}
    if task == 'batch':
        out = {'bytes': 0, 'flops': 0}
        for nx, ny in _plate_sizes(case):
            nodes, elems = (nx + 1) * (ny + 1), 2 * nx * ny
            out['bytes'] += 36 * elems + 16 * nodes + 7 * 36 * nodes + 48 * nodes
            out['flops'] += 216 * elems + 56 * nodes
        return out
    if task == 'modal':
        w = _solve_work('cube', case['n'])
        nodes = _counts('cube', case['n'])[0]
        return {'bytes': case['variants'] * (w['bytes'] + 2 * 24 * nodes * case['modes']),
                'flops': case['variants'] * w['flops'] * case['modes']}
    if task == 'train':
        nodes, _, blocks = _counts('cube', case['n'])
        weights = 8 * 64 + 2 * 32 * 64 + 96
        return {'bytes': 76 * blocks + 4 * 24 * nodes, 'flops': 3 * 2 * weights * nodes}
    problem, n = case['problem'], case['n']
    nodes, elems, blocks = _counts(problem, n)
    d = {'cube': 3, 'plate': 2, 'magnetic': 1}[problem]
    if task == 'solve':
        return _solve_work(problem, n)
    if task == 'assemble':
        npe = 4 if problem == 'cube' else 3
        return {'bytes': _mesh_bytes(problem, n) + 8 * d * d * blocks,
                'flops': (6 if case['what'] == 'stiffness' else 2) * (npe * d) ** 2 * elems}
    per = {'cube': 13, 'plate': 7, 'magnetic': 2}[problem]
    return {'bytes': _mesh_bytes(problem, n) + 8 * d * nodes + 8 * per * elems,
            'flops': {'cube': 200, 'plate': 60, 'magnetic': 20}[problem] * elems}


# ------------------------------------------------------------------------------------------------
# exact: the same values from plain torch in 64 bits
# ------------------------------------------------------------------------------------------------
def _dev():
    return 'cuda' if torch.cuda.is_available() else 'cpu'


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev())


def _gradients(coords, conn):
    """(shape-function gradients [E, npe, dim], unsigned measure [E]) of linear simplices."""
    p = _t(coords)[_t(conn).long()]
    edges = p[:, 1:] - p[:, :1]  # rows e_k
    det = torch.linalg.det(edges)
    inv = torch.linalg.inv(edges)  # column k: gradient of shape function k + 1
    g = inv.transpose(1, 2)
    g = torch.cat([-g.sum(dim=1, keepdim=True), g], dim=1)
    return g, det.abs() / math.factorial(coords.shape[1])


def _lame(problem, mats):
    E, nu = _t(mats['E']), _t(mats['nu'])
    mu = E / (2 * (1 + nu))
    lam = E * nu / ((1 + nu) * (1 - 2 * nu)) if problem == 'cube' else E * nu / (1 - nu * nu)
    return lam, mu


def _element_blocks(problem, coords, conn, mats, what):
    """[E, npe, npe, d, d] element matrices as node blocks."""
    g, vol = _gradients(coords, conn)
    npe = conn.shape[1]
    if what == 'mass':
        dim = coords.shape[1]
        rho = _t(mats['rho']) * vol * (_t(mats['thickness']) if problem == 'plate' else 1.0)
        m = (1 + torch.eye(npe, dtype=torch.float64, device=_dev())) / ((npe + 1) * npe)
        return (rho[:, None, None, None, None] * m[None, :, :, None, None] *
                torch.eye(dim, dtype=torch.float64, device=_dev())[None, None, None])
    dots = (g[:, :, None, :] * g[:, None, :, :]).sum(-1)
    if problem == 'magnetic':
        return (dots * (vol / _t(mats['mu']))[:, None, None])[..., None, None]
    lam, mu = _lame(problem, mats)
    if problem == 'plate':
        vol = vol * _t(mats['thickness'])
    outer = g[:, :, None, :, None] * g[:, None, :, None, :]
    k = (vol * lam)[:, None, None, None, None] * outer
    k += (vol * mu)[:, None, None, None, None] * outer.transpose(3, 4)
    k += ((vol * mu)[:, None, None] * dots)[..., None, None] * torch.eye(
        g.shape[2], dtype=torch.float64, device=_dev())
    return k


def _exact_blocks(problem, coords, conn, mats, what='stiffness'):
    """(row, column, value [q, d, d]) of the assembled node blocks, rows then columns ascending."""
    n = coords.shape[0]
    c = _t(conn).long()
    npe = conn.shape[1]
    key = (c[:, :, None] * n + c[:, None, :]).reshape(-1)
    keys, where = torch.unique(key, return_inverse=True)
    d = {'cube': 3, 'plate': 2, 'magnetic': 1}[problem]
    vals = torch.zeros((keys.numel(), d, d), dtype=torch.float64, device=_dev())
    blocks = max(1, 2 ** 26 // (npe * npe * d * d))
    for e0 in range(0, conn.shape[0], blocks):
        part = {k: v[e0:e0 + blocks] for k, v in mats.items()}
        ke = _element_blocks(problem, coords, conn[e0:e0 + blocks], part, what)
        vals.index_add_(0, where[e0 * npe * npe:(e0 + blocks) * npe * npe], ke.reshape(-1, d, d))
    return keys // n, keys % n, vals


class _Operator:
    """Symmetric block matrix with constrained rows and columns replaced by the identity."""

    def __init__(self, problem, coords, conn, mats, fixed, what='stiffness'):
        rows, cols, vals = _exact_blocks(problem, coords, conn, mats, what)
        d, n = vals.shape[1], coords.shape[0]
        free = torch.ones(n * d, dtype=torch.float64, device=_dev())
        free[_t(fixed)] = 0.0
        self.free, self.n, self.d = free, n * d, d
        fr = free.reshape(n, d)
        vals = vals * fr[rows][:, :, None] * fr[cols][:, None, :]
        ar = torch.arange(d, device=_dev())
        r = (rows[:, None, None] * d + ar[None, :, None]).expand_as(vals)
        c = (cols[:, None, None] * d + ar[None, None, :]).expand_as(vals)
        v = vals + ((r == c).to(torch.float64) * (1.0 - free[r]))
        self.diag = torch.zeros(n * d, dtype=torch.float64, device=_dev())
        self.diag[r[r == c]] = v[r == c]
        same = rows == cols
        self.blocks = torch.zeros((n, d, d), dtype=torch.float64, device=_dev())
        self.blocks[rows[same]] = v[same]
        self.rows, self.cols = rows, cols
        order = torch.argsort((r * (n * d) + c).reshape(-1))
        ptr = torch.zeros(n * d + 1, dtype=torch.int64, device=_dev())
        ptr[1:] = torch.cumsum(torch.bincount(r.reshape(-1), minlength=n * d), 0)
        self.csr = torch.sparse_csr_tensor(ptr, c.reshape(-1)[order], v.reshape(-1)[order],
                                           size=(n * d, n * d))

    def __matmul__(self, x):
        return (self.csr @ x[:, None])[:, 0] if x.dim() == 1 else self.csr @ x

    def solve(self, b, tol=1e-13, cap=30000):
        """Block-Jacobi conjugate gradients, restarted on the true residual."""
        inv = torch.linalg.inv(self.blocks)

        def prec(r):
            return (inv * r.reshape(-1, 1, self.d)).sum(-1).reshape(-1)

        x = torch.zeros_like(b)
        target = tol * float(b.norm())
        for _ in range(4):
            r = b - (self @ x)
            if float(r.norm()) <= target:
                break
            z = prec(r)
            p, rz = z.clone(), torch.dot(r, z)
            for it in range(cap):
                q = self @ p
                alpha = rz / torch.dot(p, q)
                x += alpha * p
                r -= alpha * q
                if it % 64 == 63 and float(r.norm()) <= 0.3 * target:
                    break
                z = prec(r)
                rz, old = torch.dot(r, z), rz
                p = z + (rz / old) * p
        return x


def exact(case, seed):
    task = case['task']
    if task == 'analysis':
        nx, ny = case['nx'], case['ny']
        pr = meshgen.cantilever_2d(nx, ny, lx=0.025 * nx, ly=0.025 * ny)
        rng = np.random.default_rng(seed)
        mats = dict(pr.materials, E=210e9 * np.exp(0.2 * rng.standard_normal(pr.conn.shape[0])))
        f = np.zeros(pr.n)
        f[2 * pr.meta['tip_node']:2 * pr.meta['tip_node'] + 2] = rng.uniform(-1e4, 1e4, 2)
        f = _t(f)
        u = _direct(_Operator('plate', pr.coords, pr.conn, mats, pr.fixed_dofs), f)
        full = _Operator('plate', pr.coords, pr.conn, mats, np.zeros(0, dtype=np.int64))
        lam = (f - (full @ u))[_t(pr.fixed_dofs)]
        return torch.cat([u, lam])
    if task == 'batch':
        out = []
        for pr in _plate_problems(case, seed):
            op = _Operator('plate', pr.coords, pr.conn, pr.materials, pr.fixed_dofs)
            out.append(_direct(op, _t(pr.f)))
        return torch.cat(out)
    if task == 'modal':
        vals = _exact_modes(case, seed)
        return None if vals is None else {'vals': vals, 'vecs': None}
    if task == 'train':
        return _exact_train(case, seed)
    kind, coords, conn, fixed = _mesh(case['problem'], case['n'], case['numbering'])
    mats = _materials(case['problem'], case['n'], coords, conn, seed)
    if task == 'solve':
        op = _Operator(case['problem'], coords, conn, mats, fixed)
        return op.solve(_t(_load(case['problem'], coords, seed)) * op.free)
    if task == 'assemble':
        rows, cols, vals = _exact_blocks(case['problem'], coords, conn, mats, case['what'])
        if case['layout'] == 'planes':
            return vals.permute(1, 2, 0).contiguous().reshape(-1)
        if case['layout'] == 'bsr':
            return vals.reshape(-1)
        # scalar CSR: within a node row, [di][block][dj]
        d = vals.shape[1]
        at = rows[:, None] * d + torch.arange(d, device=_dev())[None, :]
        order = torch.argsort(at.reshape(-1), stable=True)
        return vals.reshape(-1, d)[order].reshape(-1)
    return _exact_fields(case['problem'], coords, conn, mats, _displacement(case['problem'], coords, seed))


def _direct(op, f):
    """Dense solution of a small system, scaled to a unit diagonal first and refined twice."""
    s = op.diag.rsqrt()
    A = op.csr.to_dense() * s[:, None] * s[None, :]
    L = torch.linalg.cholesky(A)
    b = f * op.free * s
    x = torch.zeros_like(b)
    for _ in range(3):
        x = x + torch.cholesky_solve((b - (A @ x))[:, None], L)[:, 0]
    return x * s


def _exact_fields(problem, coords, conn, mats, u):
    g, vol = _gradients(coords, conn)
    d = {'cube': 3, 'plate': 2, 'magnetic': 1}[problem]
    ue = _t(u).reshape(-1, d)[_t(conn).long()]
    H = (ue[:, :, :, None] * g[:, :, None, :]).sum(1)  # du_i / dx_j
    if problem == 'magnetic':
        return [torch.stack([H[:, 0, 1], -H[:, 0, 0]]), None, None]
    lam, mu = _lame(problem, mats)
    normal = [H[:, i, i] for i in range(d)]
    shear = [H[:, 0, 1] + H[:, 1, 0]] + ([H[:, 1, 2] + H[:, 2, 1], H[:, 2, 0] + H[:, 0, 2]] if d == 3 else [])
    trace = sum(normal)
    strain = torch.stack(normal + shear)
    stress = torch.stack([lam * trace + 2 * mu * e for e in normal] + [mu * e for e in shear])
    vol = vol * _t(mats['thickness']) if problem == 'plate' else vol
    return [strain, stress, 0.5 * vol * (strain * stress).sum(0)]


def _exact_modes(case, seed):
    """Lowest eigenvalues of each draw from the dense pencil, on the host (None where that would take
    too long)."""
    kind, coords, conn, fixed = _mesh('cube', case['n'], 'grid')
    if case['n'] > 9:
        return None
    ones = {'E': np.ones(conn.shape[0]), 'nu': np.full(conn.shape[0], 0.3),
            'rho': np.full(conn.shape[0], 7850.0)}
    M = _Operator('cube', coords, conn, ones, fixed, 'mass')
    keep = torch.nonzero(M.free > 0)[:, 0].cpu()
    L = torch.linalg.cholesky(M.csr.to_dense().cpu()[keep][:, keep])
    out = []
    for E in _modal_moduli(case, seed):
        K = _Operator('cube', coords, conn, dict(ones, E=E), fixed).csr.to_dense().cpu()[keep][:, keep]
        half = torch.linalg.solve_triangular(L, K, upper=False)
        whole = torch.linalg.solve_triangular(L, half.T.contiguous(), upper=False)
        out.append(torch.linalg.eigvalsh(0.5 * (whole + whole.T))[:case['modes']])
    return torch.stack(out)


def _exact_train(case, seed):
    """Loss and gradient of the network by torch's own differentiation."""
    kind, coords, conn, fixed = _mesh('cube', case['n'], 'grid')
    op = _Operator('cube', coords, conn, _materials('cube', case['n'], coords, conn, seed), fixed)
    n, d = coords.shape[0], 3
    diag = torch.diagonal(op.blocks, dim1=1, dim2=2)
    tr = diag.sum(1).abs()
    off = op.blocks - torch.diag_embed(diag)
    deg = torch.bincount(op.rows, minlength=n).double()
    away = op.rows != op.cols
    r, c = op.rows[away], op.cols[away]
    nb = torch.bincount(r, minlength=n).double().clamp(min=1.0)

    def mean(h):
        return torch.zeros_like(h).index_add(0, r, h[c]) / nb[:, None]

    logtr = tr.log()[:, None]
    m1 = mean(logtr)
    var = (torch.zeros_like(logtr).index_add(0, r, (logtr[c] - m1[r]) ** 2) / nb[:, None])
    feat = torch.cat([logtr - m1, diag.abs() / tr[:, None], off.square().sum((1, 2)).sqrt()[:, None] / tr[:, None],
                      (1.0 - op.free).reshape(n, d).sum(1, keepdim=True) / d, deg[:, None] / 16.0, var.sqrt()],
                     dim=1)
    z = np.load(_WEIGHTS, allow_pickle=False)
    w = _t(z['params'].astype(np.float64)).requires_grad_(True)
    h, at = feat, 0
    for layer in range(3):
        fin = h.shape[1]
        W1, W2 = (w[at + k * 32 * fin:at + (k + 1) * 32 * fin].reshape(32, fin) for k in (0, 1))
        b = w[at + 64 * fin:at + 64 * fin + 32]
        at += 64 * fin + 32
        h = torch.relu(h @ W1.T + mean(h) @ W2.T + b)
    o = h @ w[at:at + 32 * d].reshape(d, 32).T + w[at + 32 * d:]
    s = torch.exp(o.clamp(-4.0, 4.0))
    inv = torch.linalg.inv(op.blocks)
    total = 0.0
    for e in _train_errors(coords, fixed, seed):
        e = _t(e)
        res = op @ e
        zz = (s * (inv * (s * res.reshape(n, d))[:, None, :]).sum(-1)).reshape(-1)
        rows = torch.dot(res, zz)
        # z . A z through the gradient of the quadratic form, which needs no sparse derivative
        az = op @ zz.detach()
        quad = 2 * torch.dot(zz, az) - torch.dot(zz.detach(), az)
        total = total + 1.0 - rows * rows / (quad * torch.dot(res, e))
    loss = total / 2
    loss.backward()
    return {'loss': loss.detach().reshape(()), 'grad': w.grad}
