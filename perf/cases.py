"""Performance cases of the framework: the calls that a user's program makes, over the ranges that it meets.

A case is a dict of plain values.  `call` names the entry point:

  bfe     batch fitness evaluation (pgh_bfe_eval) of n decision vectors
  grad    batched gradient with fitness in the same pass (pgh_batch_gradient)
  fnds    fast_non_dominated_sorting: run, sizes and every output (pgh_fnds_run / _sizes / _copy)
  sort    sort_population_mo
  select  select_best_N_mo, N = n / 2
  seed    batch_random_decision_vector (std::mt19937 draws)
  pso     one pso_gen::evolve call on a host population (pgh_pso_gen_evolve_host)
  archi   one evolve call of a device archipelago and the read-back of every island

Run from the repository root.
"""
import ctypes
import math

import numpy as np
import torch

import pagmo2_amd as P
from pagmo2_amd.workloads import archipelago_islands

KINDS = {"rosenbrock": P.ROSENBROCK, "rastrigin": P.RASTRIGIN, "ackley": P.ACKLEY, "schwefel": P.SCHWEFEL,
         "griewank": P.GRIEWANK, "lennard_jones": P.LENNARD_JONES, "zdt": P.ZDT, "dtlz": P.DTLZ}
BOUNDS = {"rosenbrock": (-5.0, 10.0), "rastrigin": (-5.12, 5.12), "ackley": (-15.0, 30.0),
          "schwefel": (-500.0, 500.0), "griewank": (-600.0, 600.0), "lennard_jones": (-3.0, 3.0),
          "zdt": (0.0, 1.0), "dtlz": (0.0, 1.0)}
PI = math.pi


def listed():
    return [
        # a small island evolved by one pso_gen call with host buffers: 100 generations of 64 individuals, where
        # launches and latency count
        dict(name="pso_rosenbrock_64x10", call="pso", problem="rosenbrock", dim=10, n=64, gen=100),
        # bulk evaluation of a wide separable problem: one bfe call on a device-resident population
        dict(name="bfe_ackley_65536x1000", call="bfe", problem="ackley", dim=1000, n=65536),
        # an ordinary batch with an odd row length and a ragged row count
        dict(name="bfe_griewank_20001x99", call="bfe", problem="griewank", dim=99, n=20001),
        # pair energies of a cluster population
        dict(name="bfe_lj_48x16384", call="bfe", problem="lennard_jones", dim=48, n=16384),
        # cluster energies with forces, an odd atom count and a ragged row count
        dict(name="grad_lj_75x4001", call="grad", problem="lennard_jones", dim=75, n=4001),
        # fitness and gradient of rows of odd length, as a local refinement asks for
        dict(name="grad_rosenbrock_30001x501", call="grad", problem="rosenbrock", dim=501, n=30001),
        # multi-objective fitness of a large population of short rows
        dict(name="bfe_zdt4_4194304x30", call="bfe", problem="zdt", prob_id=4, dim=30, n=1 << 22),
        # ranking of a two-objective population, with every output of the reference's return value
        dict(name="fnds_8192x2", call="fnds", front="spheres", n=8192, m=2),
        # one selection step of a large three-objective population with duplicated rows
        dict(name="select_16384x3", call="select", front="uniform", n=16384, m=3),
        # the sort of an ordinary genetic population merged with its offspring
        dict(name="sort_200x2", call="sort", front="spheres", n=200, m=2),
        # a large initial population drawn on the device
        dict(name="seed_rastrigin_65536x1000", call="seed", problem="rastrigin", dim=1000, n=65536),
        # an archipelago of uneven islands (populations of 32 to 4096, dimensions of 10 to 500, three problems)
        # over one evolve call of 200 generations
        dict(name="archi_32x200", call="archi", islands=32, gen=200, sizes=42),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    call = rng.choice(["bfe", "bfe", "bfe", "bfe", "grad", "grad", "fnds", "sort", "select", "seed", "pso", "archi"])
    if call in ("bfe", "grad"):
        names = ["rosenbrock", "rastrigin", "lennard_jones"]
        p = rng.choice(names if call == "grad" else names + ["ackley", "schwefel", "griewank", "zdt", "dtlz"])
        if p == "lennard_jones":
            dim = rng.randint(5, 110)
            n = min(_log(rng, 64, 32768), 60_000_000 // (dim * dim))
            return dict(call=call, problem=p, dim=dim, n=n)
        if p == "zdt":
            return dict(call=call, problem=p, prob_id=rng.choice([1, 2, 3, 4, 6]), dim=rng.choice([10, 30, 30, 31]),
                        n=_log(rng, 100, 1 << 22))
        if p == "dtlz":
            m = rng.choice([2, 3, 3, 5])
            return dict(call=call, problem=p, prob_id=rng.choice([1, 2, 3, 4, 7]), dim=m + rng.choice([4, 9, 19]),
                        nobj=m, n=_log(rng, 100, 1 << 21))
        dim = _log(rng, 2, 1000)
        return dict(call=call, problem=p, dim=dim, n=_log(rng, 64, min(1 << 20, 60_000_000 // dim)))
    if call in ("fnds", "sort", "select"):
        m = rng.choice([2, 2, 3, 3, 5])
        return dict(call=call, front="spheres" if m == 2 else "uniform", n=_log(rng, 40, 16384), m=m)
    if call == "seed":
        p = rng.choice(["rosenbrock", "rastrigin", "ackley"])
        dim = _log(rng, 10, 1000)
        return dict(call=call, problem=p, dim=dim, n=_log(rng, 64, min(1 << 18, 60_000_000 // dim)))
    if call == "pso":
        return dict(call=call, problem=rng.choice(["rosenbrock", "rastrigin"]), dim=_log(rng, 5, 100),
                    n=_log(rng, 20, 1000), gen=rng.choice([20, 50, 100]))
    return dict(call=call, islands=rng.randint(4, 24), gen=rng.choice([20, 50, 100]), sizes=rng.randrange(1000))


def _nx(case):
    return 3 * case["dim"] - 6 if case.get("problem") == "lennard_jones" else case["dim"]


def _nf(case):
    return 2 if case["problem"] == "zdt" else case.get("nobj", 1)


def _gen(seed):
    return torch.Generator(device="cuda:0").manual_seed(int(seed))


def _uniform(shape, a, b, seed):
    x = torch.empty(shape, dtype=torch.float64, device="cuda:0")
    return x.uniform_(a, b, generator=_gen(seed))


def _vectors(case, seed):
    """A population in its problem's box."""
    a, b = BOUNDS[case["problem"]]
    x = _uniform((case["n"], _nx(case)), a, b, seed)
    if case["problem"] == "zdt" and case["prob_id"] == 4:
        x[:, 1:].mul_(10.0).sub_(5.0)
    return x


def _objectives(case, seed):
    n, m = case["n"], case["m"]
    if case["front"] == "spheres":
        # distances of random points to m random centres
        x, c = _uniform((n, 30), 0.0, 1.0, seed), _uniform((m, 30), 0.0, 1.0, seed + 1)
        return torch.stack([((x - c[k]) ** 2).sum(1) for k in range(m)], 1).contiguous()
    # uniform vectors, a tenth of them exact copies of others
    f = _uniform((n, m), 0.0, 1.0, seed)
    dup = n // 10
    if dup:
        f[n - dup:] = f[torch.randint(0, n - dup, (dup,), generator=_gen(seed + 1), device="cuda:0")]
    return f


def prepare(case, seed):
    call = case["call"]
    s = dict(case)
    if call in ("bfe", "grad"):
        s["x"] = _vectors(case, seed)
        s["f"] = torch.empty((case["n"], _nf(case)), dtype=torch.float64, device="cuda:0")
        if call == "grad":
            s["g"] = torch.empty_like(s["x"])
    elif call in ("fnds", "sort", "select"):
        s["objs"] = _objectives(case, seed)
        s["ws"] = P.Fnds()
        n = case["n"]
        if call == "fnds":
            # buffers of the largest counts there can be; what a result does not fill stays zero
            s["out"] = {k: torch.zeros(c, dtype=torch.int64, device="cuda:0") for k, c in
                        (("dom_count", n), ("rank", n), ("front_offsets", n + 1), ("front_items", n),
                         ("dom_offsets", n + 1), ("dom_items", n * (n - 1) // 2))}
        else:
            s["out"] = torch.empty(n, dtype=torch.int64, device="cuda:0")
    elif call == "seed":
        s["seed"] = int(seed)
        s["x"] = torch.empty((case["n"], case["dim"]), dtype=torch.float64, device="cuda:0")
    elif call == "pso":
        a, b = BOUNDS[case["problem"]]
        s["X"] = np.random.default_rng(seed).uniform(a, b, (case["n"], case["dim"]))
        s["F"] = P.bfe_eval_host(KINDS[case["problem"]], case["dim"], s["X"]).reshape(-1)
        s["prm"] = P.pso_params(gen=case["gen"], seed=int(seed) & 0x7FFFFFFF)
    else:
        islands = archipelago_islands(case["islands"], case["gen"], case["sizes"])
        for k, d in enumerate(islands):
            d["seed"] = (int(seed) * 4096 + k) & 0x7FFFFFFF
            d["algo"] = P.pso_params(gen=case["gen"], seed=d["seed"])
        s["a"] = P.Archipelago.seeded(islands)
    return s


def run(s):
    call = s["call"]
    if call == "bfe":
        P.bfe_eval(KINDS[s["problem"]], s["dim"], s["x"], s["f"], nobj=s.get("nobj", 1), prob_id=s.get("prob_id", 0),
                   alpha=100 if s["problem"] == "dtlz" else 0)
        return s["f"]
    if call == "grad":
        P.batch_gradient(KINDS[s["problem"]], s["dim"], s["x"], s["g"], s["f"])
        return {"f": s["f"], "g": s["g"]}
    if call == "fnds":
        s["ws"].run(s["objs"])
        s["ws"].sizes()
        P.check(P.lib().pgh_fnds_copy(s["ws"].h, *(ctypes.c_void_p(t.data_ptr()) for t in s["out"].values()), 0))
        return s["out"]
    if call == "sort":
        s["ws"].sort_population_mo(s["objs"], s["out"])
        return s["out"]
    if call == "select":
        return s["out"][: s["ws"].select_best_N_mo(s["objs"], s["n"] // 2, s["out"])]
    if call == "seed":
        P.batch_random_dv(KINDS[s["problem"]], s["dim"], s["n"], s["seed"], s["x"])
        return s["x"]
    if call == "pso":
        return P.pso_gen_evolve_host(KINDS[s["problem"]], s["dim"], s["X"], s["F"], s["prm"])
    s["a"].evolve()
    return [s["a"].get(k) for k in range(s["islands"])]


def work(case):
    """Bytes: every input read once, every output written once.  Flops: the FP64 operations of the closed forms, a
    transcendental counted as one."""
    call = case["call"]
    if call in ("bfe", "grad"):
        n, nx = case["n"], _nx(case)
        b = 8 * n * (nx * (2 if call == "grad" else 1) + _nf(case))
        if case["problem"] == "lennard_jones":
            pairs = n * case["dim"] * (case["dim"] - 1) // 2
            return {"bytes": b, "flops": pairs * (28 if call == "grad" else 14)}
        return {"bytes": b, "flops": n * nx * (12 if call == "grad" else 6)}
    if call in ("fnds", "sort", "select"):
        n, m = case["n"], case["m"]
        # about 2^(1-m) of the pairs of independent objectives dominate one way or the other
        items = int(n * (n - 1) // 2 / 2 ** (m - 1)) if call == "fnds" else 0
        return {"bytes": 8 * (n * m + 4 * n + items), "flops": n * (n - 1) // 2 * m}
    if call == "seed":
        return {"bytes": 8 * case["n"] * case["dim"], "flops": 12 * case["n"] * case["dim"]}
    if call == "pso":
        e = case["n"] * case["dim"]
        return {"bytes": 16 * e, "flops": 20 * e * case["gen"]}
    total, flops = 0, 0
    for d in archipelago_islands(case["islands"], case["gen"], case["sizes"]):
        lj = d["kind"] == P.LENNARD_JONES
        e = d["pop"] * (3 * d["dim"] - 6 if lj else d["dim"])
        total += e
        flops += 20 * e + (14 * d["pop"] * d["dim"] * (d["dim"] - 1) // 2 if lj else 0)
    # X, V and the memory are read and written once a generation
    return {"bytes": 48 * total * case["gen"], "flops": flops * case["gen"]}


def _exact_fitness(case, x):
    p, n, nx = case["problem"], x.shape[0], x.shape[1]
    if p == "rosenbrock":
        return (100.0 * (x[:, :-1] ** 2 - x[:, 1:]) ** 2 + (x[:, :-1] - 1) ** 2).sum(1, keepdim=True)
    if p == "rastrigin":
        return (10.0 * nx + (x * x - 10.0 * torch.cos(2 * PI * x)).sum(1, keepdim=True))
    if p == "ackley":
        s1, s2 = (x * x).sum(1, keepdim=True) / nx, torch.cos(2 * PI * x).sum(1, keepdim=True) / nx
        return -20.0 * torch.exp(-0.2 * torch.sqrt(s1)) - torch.exp(s2) + 20.0 + math.e
    if p == "schwefel":
        return 418.9828872724338 * nx - (x * torch.sin(torch.sqrt(x.abs()))).sum(1, keepdim=True)
    if p == "griewank":
        i = torch.arange(1, nx + 1, dtype=torch.float64, device=x.device).sqrt()
        return (x * x).sum(1, keepdim=True) / 4000.0 - torch.cos(x / i).prod(1, keepdim=True) + 1.0
    if p == "zdt":
        k, f1, r = case["prob_id"], x[:, 0], x[:, 1:]
        if k == 6:
            f1 = 1.0 - torch.exp(-4.0 * f1) * torch.sin(6.0 * PI * f1) ** 6
            g = 1.0 + 9.0 * (r.sum(1) / (nx - 1.0)) ** 0.25
            return torch.stack([f1, g * (1.0 - (f1 / g) ** 2)], 1)
        if k == 4:
            g = 1.0 + 10.0 * (nx - 1.0) + (r * r - 10.0 * torch.cos(4.0 * PI * r)).sum(1)
        else:
            g = 1.0 + 9.0 * r.sum(1) / (nx - 1.0)
        q = f1 / g
        h = 1.0 - q * q if k == 2 else 1.0 - torch.sqrt(q)
        if k == 3:
            h = h - q * torch.sin(10.0 * PI * f1)
        return torch.stack([f1, g * h], 1)
    # dtlz
    k, m = case["prob_id"], case["nobj"]
    y, t = x[:, : m - 1], x[:, m - 1:]
    if k == 7:
        g = 1.0 + 9.0 * t.mean(1)
        h = m - (y / (1.0 + g)[:, None] * (1.0 + torch.sin(3.0 * PI * y))).sum(1)
        return torch.cat([y, ((1.0 + g) * h)[:, None]], 1)
    if k in (1, 3):
        g = 100.0 * (t.shape[1] + ((t - 0.5) ** 2 - torch.cos(20.0 * PI * (t - 0.5))).sum(1))
    else:
        g = ((t - 0.5) ** 2).sum(1)
    if k == 1:
        a, b, scale = y, 1.0 - y, 0.5 * (1.0 + g)
    else:
        v = (y ** 100 if k == 4 else y) * (PI / 2)
        a, b, scale = torch.cos(v), torch.sin(v), 1.0 + g
    f = []
    for j in range(m):
        v = scale * a[:, : m - 1 - j].prod(1)
        f.append(v * b[:, m - 1 - j] if j else v)
    return torch.stack(f, 1)


def _exact_gradient(case, x):
    if case["problem"] == "rosenbrock":
        g = torch.zeros_like(x)
        d = x[:, 1:] - x[:, :-1] ** 2
        g[:, :-1] = -400.0 * x[:, :-1] * d - 2.0 * (1.0 - x[:, :-1])
        g[:, 1:] += 200.0 * d
        return g
    return 2.0 * x + 20.0 * PI * torch.sin(2 * PI * x)


def _exact_lj(x, with_grad):
    """4 (r^-12 - r^-6) over the pairs: atom 0 at the origin, atom 1 on the z axis, atom 2 in the yz plane."""
    n, atoms = x.shape[0], (x.shape[1] + 6) // 3
    q = torch.zeros((n, atoms, 3), dtype=torch.float64, device=x.device)
    q[:, 1, 2] = x[:, 0]
    q[:, 2, 1:] = x[:, 1:3]
    q[:, 3:] = x[:, 3:].reshape(n, atoms - 3, 3)
    f, g = torch.empty((n, 1), dtype=torch.float64, device=x.device), torch.empty_like(x) if with_grad else None
    step = max(1, 20_000_000 // (atoms * atoms))
    eye = torch.eye(atoms, dtype=torch.bool, device=x.device)
    for b in range(0, n, step):
        d = q[b:b + step, :, None, :] - q[b:b + step, None, :, :]
        r2 = (d * d).sum(3)
        r2[:, eye] = 1.0
        s = 1.0 / (r2 * r2 * r2)
        e = 4.0 * (s * s - s)
        e[:, eye] = 0.0
        f[b:b + step, 0] = e.sum((1, 2)) / 2
        if with_grad:
            w = (24.0 * (s - 2.0 * s * s) / r2)
            w[:, eye] = 0.0
            v = (w[..., None] * d).sum(2)
            g[b:b + step, 0] = v[:, 1, 2]
            g[b:b + step, 1:3] = v[:, 2, 1:]
            g[b:b + step, 3:] = v[:, 3:].reshape(v.shape[0], -1)
    return f, g


def exact(case, seed):
    """The same outputs from the closed forms.  None where every output is a whole number (fnds, sort, select) and for
    pso_gen's trajectories (pso, archi), where rounding decides which particle is a neighbourhood's best."""
    call = case["call"]
    if call == "seed":
        a, b = BOUNDS[case["problem"]]
        count = case["n"] * case["dim"]
        w = np.frombuffer(np.random.RandomState(int(seed)).bytes(8 * count), dtype="<u4").reshape(count, 2)
        r = (w[:, 0].astype(np.float64) + w[:, 1].astype(np.float64) * 2.0 ** 32) * 2.0 ** -64
        return (np.minimum(r, 1.0 - 2.0 ** -53) * (b - a) + a).reshape(case["n"], case["dim"])
    if call not in ("bfe", "grad"):
        return None
    x = _vectors(case, seed)
    if case["problem"] == "lennard_jones":
        f, g = _exact_lj(x, call == "grad")
        return {"f": f, "g": g} if call == "grad" else f
    step = max(1, 40_000_000 // x.shape[1])
    f = torch.cat([_exact_fitness(case, c) for c in x.split(step)])
    return {"f": f, "g": torch.cat([_exact_gradient(case, c) for c in x.split(step)])} if call == "grad" else f
