"""A chained plan by value, as its workgroups' stores and polls may interleave: every workgroup walks the operations at its
own pace, its stores become visible in any order but two, and what it polls is checked against what the calls one after
the other would have it read.

The two orders: a wave's stores to one word stay in order, and a workgroup's rows of operation i are stored only when all
it stored before (the rows of i - 1, the side outputs of i) is visible.  A wave's part of an input is taken in by itself, when
no word of it is empty; the workgroup whose wave stores a part of a side output does so as soon as it may."""
import numpy as np

PRO_RMSNORM, PRO_SWIGLU = 1, 2
EMPTY = 0


class Wrong(AssertionError):
    pass


def spans(op, rows_of):
    """(address, bytes) of an operation's inputs x, b, add and of its outputs (prologue's, its sum, quantised, segments)."""
    n = op["cols"] * 4
    reads = dict(x=op["d_x"], b=op.get("d_b") if op.get("kind") else None, add=op.get("d_add"))
    writes = [op.get("d_pro_out"), op.get("d_sum_out"), op.get("d_act_out")]
    sizes = [n, n, op["cols"] // 256 * 292]
    out = [(a, s) if a else None for a, s in zip(writes, sizes)]
    return ({k: (a, n) for k, a in reads.items() if a}, out + [(d, r * 4) for d, r in rows_of(op)])


class Sim:
    def __init__(self, ops, draft, base, cells, rows_of, rng):
        self.ops, self.draft, self.base, self.rng = ops, draft, base, rng
        self.io = [spans(op, rows_of) for op in ops]
        self.user = -1 - np.arange(cells, dtype=np.int64)
        n = draft["set_bytes"] // 4
        self.slots = np.zeros(2 * n, np.int64)
        self.launches = 0

    def cell(self, addr):
        assert (addr - self.base) % 4 == 0
        return (addr - self.base) // 4

    def value(self, i, w, n):
        return ((self.launches * len(self.ops) + i) * 8 + w + 1 << 20) + np.arange(n, dtype=np.int64)

    def slot(self, at, par, other=False):
        at = at - 4 ^ (1 if other else 0)
        flip = (at ^ ((at >> 1) & par)) & 1
        return (at & ~3) // 4 + (self.draft["set_bytes"] // 4 if flip else 0)

    def in_order(self):
        """The calls one after the other: what each reads, and the memory they leave."""
        mem, want = self.user.copy(), []
        for i, (reads, writes) in enumerate(self.io):
            want.append({k: mem[self.cell(a):self.cell(a) + n // 4].copy() for k, (a, n) in reads.items()})
            for w, sp in enumerate(writes):
                if sp:
                    mem[self.cell(sp[0]):self.cell(sp[0]) + sp[1] // 4] = self.value(i, w, sp[1] // 4)
        return want, mem

    # ── a launch ──

    def launch(self):
        want, after = self.in_order()
        d, rng, G = self.draft, self.rng, self.draft["grid"]
        par = self.launches & 1
        pending = [[] for _ in range(G)]                    # per workgroup: (memory, first cell, values)

        def put(g, mem, first, values):
            cut = int(rng.integers(0, len(values) + 1))     # a store in two pieces at most
            for lo, hi in ((0, cut), (cut, len(values))):
                if hi > lo:
                    pending[g].append((mem, first + lo, values[lo:hi]))

        def settle(g, k):
            for _ in range(min(k, len(pending[g]))):
                mem, first, values = pending[g].pop(int(rng.integers(len(pending[g]))))
                mem[first:first + len(values)] = values

        def side(g, i, w, lo, hi):
            """wave stores its words lo..hi of side output w"""
            sp = self.io[i][1][w]
            if not sp:
                return
            v = self.value(i, w, sp[1] // 4)[lo:hi]
            at = 0 if w == 2 else d["ops"][i]["slot"]["pro_out" if w == 0 else "sum_out"]
            if at:
                put(g, self.slots, self.slot(at, par) + lo, v)
                put(g, self.slots, self.slot(at, par, True) + lo, np.zeros(hi - lo, np.int64))
            put(g, self.user, self.cell(sp[0]) + lo, v)

        def workgroup(g):
            for i, op in enumerate(self.ops):
                reads, writes = self.io[i]
                o = d["ops"][i]
                blocks = op["cols"] // 256
                per = 1 if blocks <= 16 else 4
                parts = [(w, w * per, min((w + 1) * per, blocks)) for w in range(16) if w * per < blocks]
                rms = op.get("kind") == PRO_RMSNORM
                mine = [p for p in parts if g + 1 + p[0] == G or (G <= p[0] and g == 0)]
                todo = [parts[k] for k in rng.permutation(len(parts))]

                def store_sides(p):
                    for w in (0, 1, 2):
                        unit = 73 if w == 2 else 256
                        side(g, i, w, p[1] * unit, p[2] * unit)
                while todo:
                    left = []
                    for p in todo:
                        lo, hi, got = p[1] * 256, p[2] * 256, {}
                        for k, (a, _) in reads.items():
                            bit = dict(x=1, add=2, b=4)[k]
                            if o["wait"] & bit:
                                first = self.slot(o["slot"][k], par)
                                got[k] = self.slots[first + lo:first + hi].copy()
                            else:
                                got[k] = self.user[self.cell(a) + lo:self.cell(a) + hi].copy()
                        if any((got[k] == EMPTY).any() for k in got):
                            left.append(p)
                            continue
                        for k in got:
                            if not np.array_equal(got[k], want[i][k][lo:hi]):
                                raise Wrong("operation %d reads another %s" % (i, k))
                        if not rms and p in mine:
                            store_sides(p)
                    if len(left) == len(todo):
                        yield "stuck"
                    elif left or rng.random() < 0.5:
                        yield "on"
                    todo = left
                if rms:
                    for p in mine:
                        store_sides(p)
                yield "on"
                while pending[g]:                           # acknowledged before the rows go out
                    settle(g, len(pending[g]))
                for k in range(len(writes) - 3):
                    first_wg = o["begin"][k]
                    last_wg = o["begin"][k + 1] if k + 4 < len(writes) else o["n_wg"]
                    if not first_wg <= g < last_wg:
                        continue
                    n, wgs, m = writes[3 + k][1] // 4, last_wg - first_wg, g - first_wg
                    lo = m * (n // wgs) + min(m, n % wgs)
                    hi = lo + n // wgs + (1 if m < n % wgs else 0)
                    v = self.value(i, 3 + k, n)[lo:hi]
                    if o["seg_slot"][k]:
                        put(g, self.slots, self.slot(o["seg_slot"][k], par) + lo, v)
                        put(g, self.slots, self.slot(o["seg_slot"][k], par, True) + lo, np.zeros(hi - lo, np.int64))
                    put(g, self.user, self.cell(writes[3 + k][0]) + lo, v)
                yield "on"
            while pending[g]:
                settle(g, len(pending[g]))

        procs = {g: workgroup(g) for g in range(G)}
        pace = rng.exponential(size=G) ** 2 + 1e-3          # some far ahead, some far behind
        lazy = rng.random(G) ** 2                           # how soon a workgroup's stores are seen
        stuck = set()                                       # polled in vain since anything was last seen
        while procs:
            if rng.random() < 0.01 or len(stuck) > len(procs) // 2:
                pace, lazy = rng.exponential(size=G) ** 2 + 1e-3, rng.random(G) ** 2
            live = [g for g in procs if g not in stuck] or list(procs)
            p = pace[live]
            g = live[int(rng.choice(len(live), p=p / p.sum()))]
            try:
                if next(procs[g]) == "stuck":
                    stuck.add(g)
                else:
                    stuck.clear()
            except StopIteration:
                del procs[g]
                stuck.clear()
            h = int(rng.integers(G))
            if pending[h] and (rng.random() < lazy[h] + 0.02 or len(stuck) == len(procs)):
                settle(h, 1 + int(rng.integers(4)))
                stuck.clear()
            if procs and len(stuck) == len(procs) and not any(pending):
                raise Wrong("everybody waits")
        if not np.array_equal(self.user, after):
            raise Wrong("the memory left behind")
        self.launches += 1


BASE, WEIGHTS = 1 << 40, 1 << 50
DIMS = (256, 512, 4352)                     # 4352: more than sixteen blocks


def rows_of(op):
    return op["rows"]


def meet(a, b):
    return a[0] < b[0] + b[1] and b[0] < a[0] + a[1]


def random_chain(rng, make_segments):
    """A few layers of a random template of dependent operations, as the dicts matvec.Plan takes (addresses of no memory),
    and the words they lie in; None where an operation's own spans meet.  Inputs are results, parts of results, prologues'
    outputs and sums, of this layer or the one before, or constants, some of which later operations store over; outputs have
    one to three places used in turn, some of them another output's."""
    top = [BASE]

    def new(n):
        at = top[0] + 4 * int(rng.integers(0, 4))
        top[0] = at + 4 * n + 80
        return at

    n_t, layers = int(rng.integers(2, 6)), int(rng.integers(1, 5))
    dims = DIMS[:2] if rng.random() < 0.8 else (DIMS[0], DIMS[2])
    rows = [[int(rng.choice(dims) if rng.random() < 0.85 else rng.choice([64, 300, 520, 768]))
             for _ in range(int(rng.choice([1, 1, 1, 2, 3])))] for _ in range(n_t)]
    norm, acts, const = new(max(dims)), [new(18 * 73) for _ in range(2)], {c: new(c) for c in dims}
    places, latest, template, ops = {}, {}, [None] * n_t, []

    def place(key, n, layer):
        if key not in places:
            others = list(places.values())
            shared = others and rng.random() < 0.12
            places[key] = ([int(rng.choice(others[int(rng.integers(len(others)))]))] if shared else
                           [new(n) for _ in range(int(rng.choice([1, 1, 2, 2, 3])))])
        return places[key][layer % len(places[key])]

    for layer in range(layers):
        for k in range(n_t):
            if layer == 0:
                later = {(j, s): n for j in range(k, n_t) for s, n in enumerate(rows[j]) if n in dims}

                def choose(least):
                    early, late = [x for x in latest if latest[x][1] >= least], [x for x in later if later[x] >= least]
                    r = rng.random()
                    if early and r < 0.8:
                        return early[-1 - min(int(rng.geometric(0.6)) - 1, len(early) - 1)]
                    return late[int(rng.integers(len(late)))] if late and r < 0.95 else None
                x = choose(min(dims))
                n = latest[x][1] if x in latest else later.get(x)
                c = int(rng.choice([d for d in dims if n is None or d <= n]))
                part = 0 if n in (None, c) or rng.random() < 0.5 else int(rng.integers(0, n - c + 1))
                kind = str(rng.choice(["none", "none", "rms", "add", "add", "swiglu"]))
                template[k] = (x, part, c, kind, choose(c) if kind in ("add", "swiglu") else None, rng.random() < 0.5,
                               rng.random() < 0.7, int(rng.choice([-1, -1, 0, 1])))
            x, part, c, kind, y, out, total, act = template[k]

            def addr(key):
                if key is None:
                    return const[c]
                return latest[key][0] if key in latest else place(key, rows[key[0]][key[1]], -1)
            op = dict(qtype=13, cols=c, d_x=addr(x) + 4 * part)
            if kind != "none":
                op.update(kind=PRO_SWIGLU if kind == "swiglu" else PRO_RMSNORM, d_b=addr(y) if kind == "swiglu" else norm)
                if out:
                    op["d_pro_out"] = place((k, "out"), c, layer)
            if kind == "add":
                op["d_add"] = addr(y)
                if total:
                    op["d_sum_out"] = place((k, "sum"), c, layer)
            if act >= 0:
                op["d_act_out"] = acts[act]
            op["rows"] = [(place((k, s), n, layer), n) for s, n in enumerate(rows[k])]
            op["segs"] = make_segments([(WEIGHTS, a, n, 0) for a, n in op["rows"]])
            reads, writes = spans(op, rows_of)
            writes = [w for w in writes if w]
            if any(meet(w, r) for w in writes for r in reads.values()) or \
               any(meet(writes[i], writes[j]) for i in range(len(writes)) for j in range(i)):
                return None
            ops.append(op)
            for key, name in (((k, "out"), "d_pro_out"), ((k, "sum"), "d_sum_out")):
                if name in op:
                    latest[key] = (op[name], c)
            latest.update({(k, s): (a, n) for s, (a, n) in enumerate(op["rows"])})
    return ops, (top[0] - BASE) // 4 + 9000
