"""Performance cases: what users of the engine have it do, through its public
entry points, from a 16 KiB buffer to 64 MiB, one automaton to 1,024.

Kinds of case:
  run    a resident input scanned again: Engine.run + Engine.reports
  scan   a new host buffer: Engine.set_input + run + reports
  load   a new rule set: Engine.load_groups, then a scan of a first buffer
  serve  requests queued at once in the request server, all of them drained
  pairs  schedule prediction: MLP.predict_pairs over (automaton, window) pairs
  train  the predictor trained on traces: MLP.train from fresh weights

Rule sets follow the workloads of ngap_amd.synth (tries of patterns of 6..40
positions, 60 % literal bytes, 30 % classes of 2..32 bytes, 10 % classes
repeated {1,4}; some automata behind a leading dot-star), drawn with numpy so
that millions of states take seconds.  A rule set is fixed by the case (a user
keeps it loaded); buffers, requests and traces come from the seed.
"""
import functools
import math

import numpy as np

from ngap_amd import Engine
from ngap_amd.groups import Group
from ngap_amd.mlp import MLP
from ngap_amd.serve import Server

KIB, MIB = 1 << 10, 1 << 20
MLP_IN, MLP_HID, WINDOW = 264, 64, 4096
ALPHABETS = {"bytes": np.arange(256), "acgt": np.frombuffer(b"ACGT", np.uint8),
             "text": np.frombuffer(b" etaoinshrdlucmfwygpbvkxjqz", np.uint8)}


# ---- rule sets ----

class Rules:
    """Automata (Group each) and what planting pattern instances needs: each
    state's predecessor on its pattern (-1 = pattern start) and its class."""

    def __init__(self, groups, prev, cls, members, count, report, owner):
        self.groups, self.prev, self.cls = groups, prev, cls
        self.members, self.count, self.report, self.owner = members, count, report, owner
        self.states = sum(g.num_states for g in groups)
        self.edges = sum(g.num_edges for g in groups)

    def plant(self, rng, data, n, group=None):
        """Writes n instances of patterns into data, at uniform positions."""
        ends = self.report if group is None else self.report[self.owner[self.report] == group]
        n = min(n, len(data))
        if n == 0 or len(ends) == 0:
            return
        s = rng.choice(ends, n)
        at = rng.integers(0, len(data), n)
        while s.size:  # one step per pattern position, last position first
            c = self.cls[s]
            data[at] = self.members[c, rng.integers(0, 1 << 30, s.size) % self.count[c]]
            s = self.prev[s]
            live = (s >= 0) & (at > 0)
            s, at = s[live], at[live] - 1


def _classes(rng, symbols, widest):
    """Class table: one class per symbol, then 4,096 of 2..widest symbols, then
    the class of all bytes.  (member table, member counts, bitmaps)"""
    k = len(symbols)
    wide = np.argsort(rng.random((4096, k)), axis=1)[:, :widest]
    members = np.zeros((k + 4097, 256), np.uint8)
    members[:k] = symbols[:, None]
    members[k:k + 4096, :wide.shape[1]] = symbols[wide]
    members[-1] = np.arange(256)
    count = np.ones(k + 4097, np.int64)
    count[k:k + 4096] = rng.integers(2, wide.shape[1] + 1, 4096)
    count[-1] = 256
    on = np.arange(256)[None, :] < count[:, None]
    bits = np.zeros((k + 4097, 256), bool)
    bits[np.nonzero(on)[0], members[on]] = True
    sets = np.packbits(bits, axis=1, bitorder="little").view("<u4").astype(np.uint32)
    return members, count, sets


@functools.lru_cache(maxsize=3)
def rules(seed, automata, lo, hi, alphabet="bytes", shortest=6, longest=40, dotstar=0.2,
          anchored=0.0, literal=0.6):
    """`automata` automata of log-uniform lo..hi states (about)."""
    rng = np.random.default_rng(seed)
    symbols = ALPHABETS[alphabet]
    k = len(symbols)
    members, count, sets = _classes(rng, symbols, min(32, max(2, k - 1)))
    size = np.exp(rng.uniform(np.log(lo), np.log(hi + 1e-9), automata))
    star = rng.random(automata) < dotstar
    # patterns per automaton, spread over its tries (about eight patterns each;
    # behind a dot-star, three tries)
    npat = np.maximum(1, np.round(size / (0.8 * (shortest + longest) / 2))).astype(np.int64)
    ntrie = np.where(star, np.minimum(npat, 3), np.maximum(1, npat // 8))
    g = np.repeat(np.arange(automata), ntrie)          # automaton of each node of the level
    w = npat[g] // ntrie[g] + (rng.random(g.size) < (npat % ntrie / ntrie)[g])
    w = np.maximum(w, 1)                               # patterns through the node
    parent, trie = np.full(g.size, -1), np.arange(g.size)
    root_anchored = rng.random(g.size) < anchored
    levels, base = [], 0
    for depth in range(1, longest + 1):                # one level of every trie at a time
        kind = rng.random(g.size)
        c = np.where(kind < literal, rng.integers(0, k, g.size), k + rng.integers(0, 4096, g.size))
        rep = (kind >= 0.9) & (literal < 1.0) & (depth > 1)
        if depth == 1:
            c = rng.integers(0, k, g.size)             # patterns start with a literal
        done = np.zeros(g.size, np.int64)
        if depth >= shortest:
            done = rng.binomial(w, 1.0 / (longest - depth + 1))
        left = w - done
        levels.append((g, parent, trie, c, rep, done > 0, np.full(g.size, depth)))
        kids = np.minimum(left, 1 + rng.binomial(np.where(rep, 2, 3), 0.25, g.size))
        ids = base + np.arange(g.size)
        base += g.size
        of = np.repeat(np.arange(g.size), kids)
        nth = np.arange(of.size) - np.repeat(np.cumsum(kids) - kids, kids)
        w = left[of] // kids[of] + (nth < left[of] % kids[of])
        g, parent, trie = g[of], ids[of], trie[of]
        if g.size == 0:
            break
    g, parent, trie, c, rep, end, depth = (np.concatenate(x) for x in zip(*levels))
    # states: a node is one state, a repeated class four; automaton by
    # automaton, trie by trie, breadth first (each dot-star state leads)
    order = np.lexsort((depth, trie, g))
    width = np.where(rep, 4, 1)[order]
    lead = np.cumsum(star)[g[order]]                   # dot-star states up to this automaton's
    first = np.empty(g.size, np.int64)
    first[order] = np.cumsum(width) - width + lead
    n = int(width.sum() + star.sum())
    star_state = np.full(automata, -1)
    nodes_before = np.zeros(automata + 1, np.int64)
    np.add.at(nodes_before, g + 1, np.where(rep, 4, 1))
    start = np.cumsum(nodes_before) + np.concatenate([[0], np.cumsum(star)])
    star_state[star] = start[:-1][star]
    owner = np.repeat(np.arange(automata), np.diff(start))
    cls = np.full(n, k + 4096, np.int64)
    prev = np.full(n, -1, np.int64)
    attrs = np.zeros(n, np.uint8)
    last = first + np.where(rep, 3, 0)
    src, dst = [], []
    for j in range(4):
        has = rep if j else np.ones(g.size, bool)
        s = first[has] + j
        cls[s] = c[has]
        attrs[s[end[has]]] |= 2
        if j:
            prev[s] = s - 1
            src.append(s - 1)
            dst.append(s)
        up = (parent >= 0) & (rep[parent] if j else True)
        src.append(first[parent[up]] + j)
        dst.append(first[up])
    inner = parent >= 0
    prev[first[inner]] = last[parent[inner]]
    root = ~inner
    starred = root & star[g]
    src += [star_state[g[starred]], star_state[star]]
    dst += [first[starred], star_state[star]]
    anch = np.zeros(g.size, bool)
    anch[root] = root_anchored[trie[root]]
    attrs[first[root & ~star[g] & ~anch]] |= 1
    attrs[star_state[star]] |= 1
    sod = np.zeros(n, bool)
    sod[first[root & ~star[g] & anch]] = True
    key = np.sort(np.concatenate(src) * n + np.concatenate(dst))
    src, dst = key // n, key % n
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))])
    words = sets[cls]
    groups = []
    for i in range(automata):
        a, b = int(start[i]), int(start[i + 1])
        groups.append(Group((row[a:b + 1] - row[a]).astype(np.int32),
                            (dst[row[a]:row[b]] - a).astype(np.int32),
                            np.ascontiguousarray(words[a:b].reshape(-1)), attrs[a:b].copy(),
                            np.nonzero(attrs[a:b] & 1)[0].astype(np.int32),
                            np.nonzero(sod[a:b])[0].astype(np.int32)))
    return Rules(groups, prev, cls, members, count, np.nonzero(attrs & 2)[0], owner)


def rules_of(case, seed=None):
    return rules(case["rules_seed"] if seed is None else seed, case["automata"], case["lo"],
                 case["hi"], case["alphabet"], case["shortest"], case["longest"],
                 case["dotstar"], case["anchored"], case["literal"])


# ---- inputs ----

def zipf_table(s, symbols):
    """2^16 symbols whose uniform choice is Zipf(s) over `symbols`."""
    p = np.arange(1, len(symbols) + 1, dtype=np.float64) ** -s
    cuts = np.round(np.cumsum(p / p.sum()) * 65536).astype(np.int64)
    return np.repeat(symbols, np.diff(np.concatenate([[0], cuts]))).astype(np.uint8)


def buffer(rng, case, R, n, chunk, group=None):
    """n bytes: iid ACGT, text-like letters, or Zipf bytes whose exponent
    drifts from chunk to chunk (0.8 .. 1.6), with planted pattern instances."""
    symbols = ALPHABETS[case["alphabet"]]
    if case["alphabet"] == "acgt":
        data = symbols[rng.integers(0, 4, n)]
    elif case["alphabet"] == "text":
        data = zipf_table(0.8, symbols)[rng.integers(0, 65536, n, dtype=np.uint16)]
    else:
        data = np.empty(n, np.uint8)
        tables = [zipf_table(1.2 - 0.4 * math.cos(2 * math.pi * i / 16), symbols)
                  for i in range(16)]
        step = max(1, n // 128) if chunk >= n else chunk * max(1, n // chunk // 128)
        for i, a in enumerate(range(0, n, step)):
            m = min(step, n - a)
            data[a:a + m] = tables[i % 16][rng.integers(0, 65536, m, dtype=np.uint16)]
    R.plant(rng, data, int(case["planted"] * n), group)
    return data


def run_options(case):
    """What the benchmark's batched engine runs with, or the library's defaults."""
    if case["schedule"] == "plain":
        return dict(algorithm="nonblockingallgroups", unique=bool(case["unique"]))
    return dict(algorithm="nonblockingallgroups", schedule="batched",
                precompute_depth=case["depth"], unique=bool(case["unique"]),
                active_threshold=0, fallback=True)


def traces(rng, windows, automata):
    """Features of windows x automata: normalised byte histograms of 4 KiB
    windows and automaton statistics (log sizes, mean degree, shares)."""
    hist = np.empty((windows, 256), np.float32)
    tables = [zipf_table(s, np.arange(256)) for s in (0.8, 1.0, 1.2, 1.4, 1.6)]
    for a in range(0, windows, 64):
        m = min(64, windows - a)
        b = tables[(a // 64) % 5][rng.integers(0, 65536, m * WINDOW, dtype=np.uint16)]
        of = np.repeat(np.arange(m, dtype=np.int64) * 256, WINDOW) + b
        hist[a:a + m] = np.bincount(of, minlength=m * 256).reshape(m, 256) / np.float32(WINDOW)
    n = np.exp(rng.uniform(np.log(50), np.log(50000), automata))
    stats = np.stack([np.log1p(n), np.log1p(n * 1.2), np.log1p(n / 100), 0 * n, np.log1p(n / 20),
                      rng.uniform(1.0, 1.4, automata), rng.uniform(0, 0.02, automata),
                      np.log1p(rng.random(automata) < 0.2)], 1).astype(np.float32)
    return hist, stats


def weights(rng):
    """Fresh predictor weights: He-uniform matrices, zero biases."""
    def he(a, b):
        return rng.uniform(-1, 1, a * b) * math.sqrt(6.0 / a)

    return np.concatenate([he(MLP_IN, MLP_HID), np.zeros(MLP_HID), he(MLP_HID, MLP_HID),
                           np.zeros(MLP_HID), he(MLP_HID, 1), np.zeros(1)]).astype(np.float32)


def train_data(rng, case):
    """Traces as the benchmark samples them: (automaton, window) features and
    log item counts, roughly linear in the features plus noise."""
    hist, stats = traces(rng, 512, 256)
    w, g = rng.integers(0, 512, case["n"]), rng.integers(0, 256, case["n"])
    x = np.concatenate([hist[w], stats[g]], 1)
    t = 0.6 * stats[g, 0] + 8 * hist[w, 0] + 0.2 * rng.standard_normal(case["n"])
    return dict(x=x, t=t.astype(np.float32), weights=weights(rng))


# ---- the cases ----

RULES = dict(alphabet="bytes", shortest=6, longest=40, dotstar=0.2, anchored=0.0, literal=0.6,
             planted=1e-4, schedule="batched", depth=3, unique=True)


def listed():
    def rule_case(name, kind, automata, lo, hi, size, chunk, **kw):
        return dict(dict(RULES, name=name, kind=kind, rules_seed=1, automata=automata, lo=lo,
                         hi=hi, size=size, chunk=chunk), **kw)

    acgt = dict(alphabet="acgt", shortest=8, longest=16, dotstar=0.0, literal=1.0)
    return [
        # a small buffer against 64 DNA literals, the whole call: all latency
        rule_case("scan_literal_16k", "scan", 1, 770, 770, 16 * KIB, 16 * KIB, **acgt),
        # the benchmark's DNA literal workload, input resident, one chunk
        rule_case("run_literal_1m", "run", 1, 770, 770, MIB, MIB, **acgt),
        # one large regex automaton over 16 MiB in 256 KiB chunks
        rule_case("run_regex_16m", "run", 1, 400000, 400000, 16 * MIB, 256 * KIB, dotstar=0.0),
        # the headline workload: 1,024 automata, drifting bytes, 8 MiB in 64 KiB
        rule_case("run_rules_8m", "run", 1024, 50, 50000, 8 * MIB, 64 * KIB),
        # the same rule set over a large resident input
        rule_case("run_rules_64m", "run", 1024, 50, 50000, 64 * MIB, 64 * KIB),
        # network-style scan of a new buffer: ragged chunks, anchored patterns,
        # shallow memo tables (depth 2)
        rule_case("scan_rules_ragged", "scan", 200, 50, 20000, 131 * 50021, 50021, depth=2,
                  anchored=0.1),
        # text against short words: matches everywhere, the report path
        rule_case("run_words_dense_4m", "run", 8, 300, 3000, 4 * MIB, 64 * KIB, alphabet="text",
                  shortest=3, longest=12, dotstar=0.1, literal=0.9),
        # the library's default options: one workgroup per (group, chunk), no
        # memo tables beyond single bytes
        rule_case("run_default_1m", "run", 4, 20000, 20000, MIB, 16 * KIB, schedule="plain",
                  depth=1, unique=False),
        # a new rule set compiled into the device image, then a first buffer
        rule_case("load_rules", "load", 128, 500, 50000, MIB, 64 * KIB),
        # requests of 1 KiB .. 1 MiB on 64 resident automata, queued at once
        rule_case("serve_mix", "serve", 64, 1000, 100000, 192, 0, smallest=KIB, biggest=MIB),
        # predicted cost of every (automaton, 4 KiB window) of an 8 MiB input
        dict(name="predict_pairs_2m", kind="pairs", automata=1024, windows=2048, every=True,
             n=2097152),
        # the predictor trained on 65,536 traces, mini-batches as the benchmark's
        dict(name="train_64k", kind="train", n=65536, epochs=2, batch=4096),
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["run", "run", "run", "scan", "scan", "dense", "plain", "load", "serve",
                       "pairs", "train"])
    if kind == "pairs":
        n = log(1000, 2000000)
        return dict(kind="pairs", automata=log(8, 1024), windows=log(16, 2048), every=False, n=n)
    if kind == "train":
        return dict(kind="train", n=log(2000, 60000), epochs=rng.randint(1, 2),
                    batch=log(256, 4096))
    case = dict(RULES, kind=kind, rules_seed=rng.randrange(1, 1 << 20))
    if kind in ("run", "scan"):
        automata = log(1, 512)
        hi = min(100000, 2000000 // automata)
        size = log(16 * KIB, 32 * MIB)
        case.update(automata=automata, lo=max(20, hi // rng.choice([1, 10, 100])), hi=hi,
                    size=size, chunk=min(size, log(2 * KIB, MIB)), depth=rng.choice([2, 3, 3]),
                    anchored=rng.choice([0.0, 0.1]), unique=rng.random() < 0.8)
    elif kind == "dense":
        case.update(kind="run", automata=log(1, 32), lo=100, hi=log(300, 3000), alphabet="text",
                    shortest=rng.randint(3, 4), longest=rng.randint(8, 12), literal=0.9, dotstar=0.1,
                    size=log(64 * KIB, 4 * MIB), chunk=log(4 * KIB, 64 * KIB),
                    depth=rng.choice([2, 3]))
    elif kind == "plain":
        case.update(kind="run", automata=log(1, 8), lo=1000, hi=log(2000, 20000),
                    schedule="plain", depth=1, unique=False, size=log(64 * KIB, MIB),
                    chunk=log(4 * KIB, 32 * KIB))
    elif kind == "load":
        automata = log(1, 256)
        case.update(automata=automata, lo=50, hi=min(50000, 1200000 // automata),
                    size=log(16 * KIB, MIB), chunk=16 * KIB, depth=rng.choice([2, 3]))
    else:
        case.update(automata=log(2, 64), lo=1000, hi=log(2000, 50000), size=log(4, 192), chunk=0,
                    smallest=log(256, 4 * KIB), biggest=log(8 * KIB, MIB))
    return case


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "pairs":
        hist, stats = traces(rng, case["windows"], case["automata"])
        if case["every"]:
            pairs = np.stack(np.meshgrid(np.arange(case["automata"]), np.arange(case["windows"]),
                                         indexing="ij"), -1).reshape(-1, 2).astype(np.uint32)
        else:
            pairs = np.stack([rng.integers(0, case["automata"], case["n"]),
                              rng.integers(0, case["windows"], case["n"])], 1).astype(np.uint32)
        p = weights(rng)
        m = MLP(0)
        m.params = p
        return dict(kind=kind, mlp=m, weights=p, hist=hist, stats=stats, pairs=pairs)
    if kind == "train":
        return dict(train_data(rng, case), kind=kind, seed=seed, case=case)
    R = rules_of(case, case["rules_seed"] + seed if kind == "load" else None)
    e = Engine(0)
    st = dict(kind=kind, engine=e, opts=run_options(case), chunk=case["chunk"])
    total = case["size"] * (case["biggest"] if kind == "serve" else 1)
    st["out"] = np.zeros(1025 + (total if case["alphabet"] == "text" else total // 256), np.int64)
    if kind == "serve":
        e.load_groups(R.groups, case["depth"])
        lens = np.exp(rng.uniform(np.log(case["smallest"]), np.log(case["biggest"]),
                                  case["size"])).astype(np.int64)
        to = rng.integers(0, case["automata"], case["size"])
        st["requests"] = [(int(g), buffer(rng, case, R, int(n), int(n), int(g)))
                          for g, n in zip(to, lens)]
        st["server"] = Server(e, max_inflight=4, **run_options(case))
        return st
    st["data"] = buffer(rng, case, R, case["size"], case["chunk"])
    if kind == "load":
        st["groups"], st["depth"] = R.groups, case["depth"]
        return st
    e.load_groups(R.groups, case["depth"])
    if kind == "run":
        e.set_input(st["data"], case["chunk"])
    return st


def fill(out, reports):
    """A pass's reports in the program's own buffer, their number first."""
    out[0] = reports.size
    out[1:1 + reports.size] = reports.view(np.int64)
    return out


def run(st):
    kind = st["kind"]
    if kind == "pairs":
        return st["mlp"].predict_pairs(st["hist"], st["stats"], st["pairs"])
    if kind == "train":
        c = st["case"]
        m = MLP(0)
        m.params = st["weights"]
        loss = m.train(st["x"], st["t"], epochs=c["epochs"], batch=c["batch"], lr=2e-3,
                       seed=st["seed"])
        out = {"params": m.params, "loss": float(loss)}
        m.close()
        return out
    if kind == "serve":
        s = st["server"]
        ids = [s.submit(g, d) for g, d in st["requests"]]
        done = s.drain(ids)
        reports = [done[i][0] for i in ids]
        return {"counts": np.array([len(r) for r in reports], np.int64),
                "reports": fill(st["out"], np.concatenate(reports))}
    e = st["engine"]
    if kind == "load":
        e.load_groups(st["groups"], st["depth"])
    if kind != "run":
        e.set_input(st["data"], st["chunk"])
    e.run(**st["opts"])
    return fill(st["out"], e.reports())


# ---- what a pass cannot do without ----

def work(case):
    """Bytes: the host or resident input once, the outputs once (reports by the
    planted instances).  Flops: the predictor's products, the first layer's
    once per window and once per automaton."""
    kind = case["kind"]
    if kind == "pairs":
        n, w, g = case["n"], case["windows"], case["automata"]
        return dict(bytes=12 * n + 1024 * w + 32 * g,
                    flops=2.0 * (n * (MLP_HID * MLP_HID + MLP_HID) + w * 256 * MLP_HID
                                 + g * 8 * MLP_HID))
    if kind == "train":
        params = MLP_IN * MLP_HID + MLP_HID * MLP_HID + MLP_HID
        # forward, weight gradients, and the second layer's input gradient
        per = 2.0 * (2 * params + MLP_HID * MLP_HID)
        return dict(bytes=4 * (MLP_IN + 1) * case["n"], flops=per * case["n"] * case["epochs"])
    if kind == "serve":
        a, b = case["smallest"], case["biggest"]
        return dict(bytes=case["size"] * (b - a) / math.log(b / a), flops=0)
    size = case["size"] // case["chunk"] * case["chunk"]
    extra = 8 * case["planted"] * size
    if kind == "load":
        states = case["automata"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        extra += states * 41  # 32 B class, 4 B row offset, 1 B flags, 4 B per edge
    return dict(bytes=size + extra, flops=0)


# ---- the predictor in 64 bits ----

def layers(p):
    """W1[264, 64], b1, W2[64, 64], b2, W3[64], b3 of the flat parameters."""
    shapes = ((MLP_IN, MLP_HID), (MLP_HID,), (MLP_HID, MLP_HID), (MLP_HID,), (MLP_HID,), (1,))
    cuts = np.cumsum([math.prod(s) for s in shapes])
    return [a.reshape(s) for a, s in zip(np.split(p, cuts[:-1]), shapes)]


def exact_pairs(st):
    W1, b1, W2, b2, W3, b3 = layers(st["weights"].astype(np.float64))
    by_window = st["hist"].astype(np.float64) @ W1[:256]
    by_automaton = st["stats"].astype(np.float64) @ W1[256:] + b1
    y = np.empty(len(st["pairs"]))
    for a in range(0, len(y), 1 << 17):
        g, w = st["pairs"][a:a + (1 << 17)].T
        h = np.maximum(np.maximum(by_window[w] + by_automaton[g], 0) @ W2 + b2, 0)
        y[a:a + (1 << 17)] = h @ W3 + b3
    return y


def exact_train(case, st, seed):
    """MLP.train in float64: Fisher-Yates with the trainer's generator, mean
    squared error, Adam."""
    p = st["weights"].astype(np.float64)
    x, t = st["x"].astype(np.float64), st["t"].astype(np.float64)
    n, batch = case["n"], case["batch"]
    lr, b1, b2, eps = (float(np.float32(v)) for v in (2e-3, 0.9, 0.999, 1e-8))
    mom, var, step, z, idx = np.zeros_like(p), np.zeros_like(p), 0, seed, list(range(n))
    for _ in range(case["epochs"]):
        for i in range(n - 1, 0, -1):
            z = (z * 6364136223846793005 + 1442695040888963407) & (2**64 - 1)
            j = (z >> 33) % (i + 1)
            idx[i], idx[j] = idx[j], idx[i]
        total = 0.0
        for a in range(0, n, batch):
            take = idx[a:a + batch]
            W1, c1, W2, c2, W3, c3 = layers(p)
            X = x[take]
            H1 = np.maximum(X @ W1 + c1, 0)
            H2 = np.maximum(H1 @ W2 + c2, 0)
            err = H2 @ W3 + c3 - t[take]
            total += float(err @ err)
            dy = 2 * err / len(take)
            d2 = np.outer(dy, W3) * (H2 > 0)
            d1 = (d2 @ W2.T) * (H1 > 0)
            grad = np.concatenate([(X.T @ d1).ravel(), d1.sum(0), (H1.T @ d2).ravel(), d2.sum(0),
                                   H2.T @ dy, [dy.sum()]])
            step += 1
            mom = b1 * mom + (1 - b1) * grad
            var = b2 * var + (1 - b2) * grad * grad
            p = p - lr * (mom / (1 - b1**step)) / (np.sqrt(var / (1 - b2**step)) + eps)
    return {"params": p, "loss": total / n}


def exact(case, seed):
    """The predictor's outputs in 64 bits.  Reports are whole numbers,
    which are compared as they are."""
    if case["kind"] == "pairs":
        return exact_pairs(prepare(case, seed))
    if case["kind"] == "train":
        return exact_train(case, train_data(np.random.default_rng(seed), case), seed)
    return None
