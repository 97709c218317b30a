"""Statement order of large kernel bodies: register pressure and load distance.

A BSSN body reads up to 440 stencil values and evaluates a thousand CSE'd statements. In
the order FD_outputC emits them (every read, every stencil, then the expressions) hundreds
of values are live at once, and the compiler's scheduler, working on one huge basic block,
neither reaches the smallest pressure nor keeps many loads in flight. ``reorder`` rewrites a
body into an order chosen here:

* Every sum is taken apart into its terms and written as an accumulation, and the terms of
  all sums are ordered by a backward greedy search: the next term (from the end of the body)
  is the one that leaves the fewest values live, counting operands that collapse into loads
  or already live values at once. A few seeded tie-breaks are tried and the order with the
  smallest peak is kept, so the result is the same on every run.
* A read is placed ``prefetch`` terms before its first use, so that loads overlap the
  arithmetic of the terms in between.
* A scheduling barrier every ``region`` terms keeps the compiler from undoing the order. With
  ``sync`` it is a workgroup barrier, which also keeps a block's waves on the same fields, so
  that the rows they share are still in the L1 cache.

The terms of a sum are added in the new order, so results agree with the plain body's to
rounding. Statements whose grouping carries precision (the differences of
FD_difference_from_centre) are kept whole.
"""
import ast
import random
import re

_DECL = re.compile(r"^(?:const )?double (\w+) = (.*);$")
_WRITE = re.compile(r"^(\w+\[.*\]) (\+?=) (.*);$")
_READ = re.compile(r"^\w+(\[[^\[\]]*\])+$")
_NAME = re.compile(r"[A-Za-z_]\w*")
# differences of stencil values (finite_difference._differenced_stencil)
_WHOLE = re.compile(r"_(p\d+|q\d\d|d\d)$")


class _Value:
    def __init__(self, kind, name, text=None):
        self.kind, self.name, self.text = kind, name, text   # kind: load, const, sum
        self.terms = []                                      # sum: (operands, sign, C text)


class _Body:
    """The values of a body as a graph: loads, constants and sums of products."""

    def __init__(self):
        self.vals, self.index, self.anonymous, self.writes = [], {}, {}, []

    def new(self, value):
        self.vals.append(value)
        return len(self.vals) - 1

    def product(self, node):
        """(operand values, C text) of an expression that is not a sum at its top."""
        if isinstance(node, ast.Name):
            v = self.index.get(node.id)
            return ([] if v is None or self.vals[v].kind == "const" else [v]), node.id
        if isinstance(node, ast.Constant):
            return [], repr(node.value)
        if isinstance(node, ast.UnaryOp) and isinstance(node.op, ast.USub):
            ops, t = self.product(node.operand)
            return ops, "(-%s)" % t
        if isinstance(node, ast.BinOp) and isinstance(node.op, (ast.Mult, ast.Div)):
            a, ta = self.product(node.left)
            b, tb = self.product(node.right)
            return a + b, "%s*%s" % (ta, tb) if isinstance(node.op, ast.Mult) else "%s/(%s)" % (ta, tb)
        if isinstance(node, ast.Call):
            parts = [self.product(a) for a in node.args]
            return [o for p, _ in parts for o in p], "%s(%s)" % (node.func.id, ", ".join(t for _, t in parts))
        if isinstance(node, ast.BinOp) and isinstance(node.op, (ast.Add, ast.Sub)):
            if not any(n.id in self.index and self.vals[self.index[n.id]].kind != "const"
                       for n in ast.walk(node) if isinstance(n, ast.Name)):
                return [], "(%s)" % ast.unparse(node)   # parameters and literals only
            v = self.sum(node)
            return [v], self.vals[v].name
        raise ValueError("schedule: unsupported expression " + ast.unparse(node))

    def _flatten(self, node, sign, out):
        if isinstance(node, ast.BinOp) and isinstance(node.op, (ast.Add, ast.Sub)):
            self._flatten(node.left, sign, out)
            self._flatten(node.right, sign if isinstance(node.op, ast.Add) else -sign, out)
        elif isinstance(node, ast.UnaryOp) and isinstance(node.op, ast.USub):
            self._flatten(node.operand, -sign, out)
        else:
            out.append((sign, node))

    def sum(self, node, name=None):
        """The value of an expression, as a sum of its terms."""
        key = ast.dump(node)
        if name is None and key in self.anonymous:
            return self.anonymous[key]
        flat = []
        self._flatten(node, 1, flat)
        terms = [(self.product(n), s) for s, n in flat]
        if name is None:
            name = "nrpy_s%d" % len(self.vals)
        v = self.new(_Value("sum", name))
        self.vals[v].terms = [(ops, s, t) for (ops, t), s in terms]
        self.anonymous.setdefault(key, v)
        return v

    def add(self, name, text):
        if "[" in text:
            if not _READ.match(text):
                raise ValueError("schedule: unsupported read " + text)
            self.index[name] = self.new(_Value("load", name, text))
            return
        operands = [self.index[n] for n in _NAME.findall(text) if n in self.index]
        if not any(self.vals[o].kind != "const" for o in operands):
            self.index[name] = self.new(_Value("const", name, text))
        elif "?" in text or _WHOLE.search(name):
            v = self.new(_Value("sum", name))
            self.vals[v].terms = [([o for o in operands if self.vals[o].kind != "const"], 1, text)]
            self.index[name] = v
        else:
            self.index[name] = self.sum(ast.parse(text.strip(), mode="eval").body, name)

    def write(self, target, op, text):
        text = text.strip()
        if text in self.index and self.vals[self.index[text]].kind != "const":
            v = self.index[text]
        else:
            v = self.sum(ast.parse(text, mode="eval").body, "nrpy_w%d" % len(self.writes))
        self.writes.append((v, target, op))


def _order(body, rng, noise):
    """(terms in execution order: (value, term index), or (load, -1); peak of live values)."""
    vals = body.vals
    rem = [0] * len(vals)                    # uses not scheduled yet, by values that a write needs
    needed, todo = set(), [v for v, _, _ in body.writes]
    while todo:
        v = todo.pop()
        if v in needed:
            continue
        needed.add(v)
        for ops, _, _ in vals[v].terms:
            for o in ops:
                rem[o] += 1
                todo.append(o)
    live, pending, stamp, order = set(), {}, {}, []
    for v, _, _ in body.writes:
        live.add(v)
        if rem[v] == 0 and vals[v].kind == "sum":
            pending[v] = list(range(len(vals[v].terms)))

    def cost(o, uses, depth=0):
        """Live values added by making o an operand of a term with `uses` of it."""
        base = 0 if o in live else 1
        if rem[o] > uses:
            return base
        if vals[o].kind == "load":
            return base - 1
        if depth > 3:
            return base
        count, c = {}, 0
        for ops, _, _ in vals[o].terms:
            for p in ops:
                count[p] = count.get(p, 0) + 1
        for p, k in count.items():
            c += cost(p, k, depth + 1)
            if c > 1:
                break
        return min(base, base - 1 + c)

    step, peak = 0, 0
    while pending:
        best = None
        for s, left in pending.items():
            for ti in left:
                count = {}
                for o in vals[s].terms[ti][0]:
                    count[o] = count.get(o, 0) + 1
                last = len(left) == 1
                key = (sum(cost(o, k) for o, k in count.items()) - last + (rng.random() * noise if rng else 0),
                       sum(o not in live for o in count) - last, len(left), -stamp.get(s, 0), s, ti)
                if best is None or key < best[0]:
                    best = (key, s, ti)
        _, s, ti = best
        step += 1
        order.append((s, ti))
        pending[s].remove(ti)
        stamp[s] = step
        if not pending[s]:
            del pending[s]
            live.discard(s)
        ops = vals[s].terms[ti][0]
        for o in ops:
            rem[o] -= 1
            live.add(o)
        peak = max(peak, len(live))
        for o in dict.fromkeys(ops):
            if rem[o] == 0:
                if vals[o].kind == "load":
                    order.append((o, -1))
                    live.discard(o)
                elif o not in pending:
                    pending[o] = list(range(len(vals[o].terms)))
                    stamp[o] = step
    order.reverse()
    return order, peak


def reorder(body, prefetch, region, sync=False, tries=4):
    """The body of a kernel (FD_outputC's block, or pass 1 of a vector-Jacobian product) in the
    order described above. Raises ValueError for statements it does not know."""
    lines = body.splitlines()
    known = [k for k, l in enumerate(lines) if _DECL.match(l.strip()) or _WRITE.match(l.strip())]
    first, last = known[0], known[-1]
    b = _Body()
    for l in lines[first:last + 1]:
        l = l.strip()
        m = _DECL.match(l)
        if m:
            b.add(m.group(1), m.group(2))
            continue
        m = _WRITE.match(l)
        if m:
            b.write(*m.groups())
        elif l and not l.startswith(("/*", "//")):
            raise ValueError("schedule: unknown statement " + l)
    best = None
    for seed in range(tries):
        order, peak = _order(b, random.Random(seed) if seed else None, 0.6)
        if best is None or peak < best[1]:
            best = (order, peak)
    return "\n".join(lines[:first] + _emit(b, best[0], prefetch, region, sync,
                                            re.match(r"\s*", lines[first]).group(0)) + lines[last + 1:]) + "\n"


def _emit(b, order, prefetch, region, sync, indent):
    vals, out = b.vals, []
    before = {}                              # term number -> loads placed in front of it
    n = 0
    for v, ti in order:
        if ti < 0:
            before.setdefault(max(0, n - prefetch), []).append(v)
        else:
            n += 1
    writes = {}
    for v, target, op in b.writes:
        writes.setdefault(v, []).append((target, op))
    used = {v for v, ti in order}
    for v in vals:
        if v.kind == "const":
            out.append("const double %s = %s;" % (v.name, v.text))
    for v in range(len(vals)):               # a write of a plain read
        if v not in used and v in writes and vals[v].kind == "load":
            before.setdefault(0, []).append(v)
    left = {v: len(vals[v].terms) for v in used}
    n = 0

    def store(v):
        for target, op in writes.get(v, ()):
            out.append("%s %s %s;" % (target, op, vals[v].name))
    for v, ti in order:
        if ti < 0:
            continue
        if region and n and n % region == 0:
            out.append("__builtin_amdgcn_s_barrier();" if sync else "__builtin_amdgcn_sched_barrier(0);")
        for l in before.get(n, ()):
            out.append("const double %s = %s;" % (vals[l].name, vals[l].text))
            store(l)
        n += 1
        ops, sign, text = vals[v].terms[ti]
        whole = len(vals[v].terms)
        if left[v] == whole:
            out.append("%sdouble %s = %s;" % ("const " if whole == 1 else "", vals[v].name,
                                              text if sign > 0 else "-(%s)" % text))
        else:
            out.append("%s %s= %s;" % (vals[v].name, "+" if sign > 0 else "-", text))
        left[v] -= 1
        if left[v] == 0:
            store(v)
    return [indent + l for l in out]
