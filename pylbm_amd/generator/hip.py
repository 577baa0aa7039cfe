"""HIP (gfx950) code generator for one lattice Boltzmann scheme.

Plays the role of pylbm's code printers + ``CodeGen`` (pylbm/generator/codegen.py:
1014-1178 for Cython, printing/cython.py:301-350) for the routines
``one_time_step`` (pylbm/algorithm/pull.py:11-59), ``f2m``, ``m2f`` and
``equilibrium`` (pylbm/algorithm/base.py:298-402): from the frozen
:class:`~pylbm_amd.scheme.KernelSpec` it prints one ``.hip`` translation unit
holding

* ``fused_step<S, FOLD>``: pull f_k(x - v_k), m = M f, [source dt/2],
  relax m_i <- (1 - s_i) m_i + s_i eq_i(m_c), [source dt/2], fnew = M^-1 m,
  one thread per interior cell, stored through the population codec S;
* ``f2m_kernel<S>`` / ``m2f_kernel<S>`` / ``equilibrium_kernel`` over the whole
  halo-inclusive domain with FP64 moments;
* the ``extern "C"`` entry points declared in include/pylbm_hip.h.

The q x q transforms are printed from the exact rational matrices.  When every
moment polynomial has a definite parity under v -> -v (true for the usual MRT
bases) the transforms are factored through the pair sums f_k + f_ksym and
differences f_k - f_ksym, which halves the work; terms sharing a coefficient
are grouped and identical partial sums are computed once.  Relaxation rates
are run-time arguments, so one compiled module serves every viscosity; only
the zero pattern of s (which rows are relaxed at all, pylbm drops identity
rows, printing/cython.py:347-349) is baked in.
"""
import hashlib
import os
import re
from fractions import Fraction

import sympy as sp
from sympy.printing.c import C99CodePrinter

from ..scheme import KernelSpec

__all__ = ["generate_source", "spec_hash"]


def _source_tag() -> str:
    """Digest of the code generator, its compile flags and the device header it
    includes: a module built from other sources never matches the cache key."""
    h = hashlib.sha1()
    here = os.path.dirname(os.path.abspath(__file__))
    for path in (os.path.abspath(__file__), os.path.join(here, "build.py"),
                 os.path.join(here, "..", "csrc", "lbm_device.h"),
                 os.path.join(here, "..", "..", "include", "pylbm_hip.h")):
        with open(path, "rb") as fh:
            h.update(fh.read())
    return h.hexdigest()[:12]


_SOURCE_TAG = _source_tag()


def spec_hash(spec: KernelSpec) -> str:
    return hashlib.sha1((spec.key() + _SOURCE_TAG).encode()).hexdigest()[:16]


def _lit(x) -> str:
    """Correctly rounded FP64 literal of an exact rational, cast to the compute type."""
    v = float(Fraction(x)) if not isinstance(x, float) else x
    r = repr(v)
    if "e" not in r and "." not in r and "inf" not in r and "nan" not in r:
        r += ".0"
    return "C(%s)" % r


class _Printer(C99CodePrinter):
    """Prints sympy expressions in the compute type ``C`` of the kernels."""

    def _print_Symbol(self, expr):
        name = expr.name
        if name == "t":
            return "tt"
        if name in ("X", "Y", "Z"):
            return "xc%d" % "XYZ".index(name)
        if name.startswith("cr") and name[2:].isdigit():
            return "cref[%s]" % name[2:]
        return name

    def _print_Integer(self, expr):
        return _lit(int(expr))

    def _print_Rational(self, expr):
        return _lit(Fraction(int(expr.p), int(expr.q)))

    def _print_Float(self, expr):
        return _lit(float(expr))

    def _print_Pow(self, expr):
        b, e = expr.as_base_exp()
        if e.is_Integer:
            n = int(e)
            if n == 0:
                return "C(1.0)"
            base = self.parenthesize(b, 100)
            prod = "*".join([base] * abs(n))
            return "(%s)" % prod if n > 0 else "(C(1.0)/(%s))" % prod
        if e == sp.Rational(1, 2):
            return "sqrt(%s)" % self._print(b)
        if e.is_number and e.is_real:
            return "pow(%s, %s)" % (self._print(b), self._print(e))
        raise NotImplementedError("power %s not supported" % expr)

    def __init__(self, fuse):
        super().__init__()
        self.fuse = fuse

    def _print_Add(self, expr, order=None):
        """With fuse the terms without a product come first: every product is then
        contracted into an FMA with the sum so far."""
        if not self.fuse:
            return super()._print_Add(expr, order=order)
        terms = self._as_ordered_terms(expr, order=order)
        plain = [t for t in terms if not (t.is_Mul and t.as_coeff_Mul()[0] != -1) and not t.is_Pow]
        rest = [t for t in terms if t not in plain]
        out = ""
        for t in plain + rest:
            text = self._print(t)
            if not out:
                out = text
            elif text.startswith("-"):
                out += " - " + text[1:]
            else:
                out += " + " + text
        return out


def _ccode(expr, fuse=True) -> str:
    return _Printer(fuse).doprint(expr)


# ----------------------------------------------------------------- structure
def _canon(v, dim):
    """Reference axes -> canonical (outer, mid, inner)."""
    v = list(v)
    return tuple([0] * (3 - dim) + v)


def _pairs(spec: KernelSpec):
    """ksym[k] inside the same block of M, or None if the stencil is not symmetric."""
    ns = spec.ns
    blocks = spec.blocks
    ksym = [None] * ns
    for lo, hi in blocks:
        index = {tuple(spec.velocities[j]): j for j in range(lo, hi)}
        for k in range(lo, hi):
            neg = tuple(-c for c in spec.velocities[k])
            if neg not in index:
                return None
            ksym[k] = index[neg]
    return ksym


def _row_parities(mat, ksym, by_rows=True):
    """Parity sigma_i of every row i (by_rows: mat[i][ksym j] == sigma_i mat[i][j]) or
    column i (mat[ksym j][i] == sigma_i mat[j][i]); None if one is indefinite."""
    ns = len(mat)
    get = (lambda i, j: mat[i][j]) if by_rows else (lambda i, j: mat[j][i])
    sig = []
    for i in range(ns):
        s = 0
        for j in range(ns):
            a = get(i, j)
            if a == 0 or ksym[j] == j:
                continue
            b = get(i, ksym[j])
            if b == a:
                s = 1
            elif b == -a:
                s = -1
            else:
                return None
            break
        s = s or 1
        for j in range(ns):
            if get(i, ksym[j]) != s * get(i, j):
                return None
        sig.append(s)
    return sig


class _SumBuilder:
    """Emits grouped linear combinations, reusing identical partial sums; with fuse also
    the common pairs of different sums, and ordered for the contraction of products."""

    def __init__(self, prefix, fuse=True):
        self.fuse = fuse
        self.sums = []      # (name, [(sign, var)])
        self.late = []      # lines that use the sums
        self.cache = {}
        self.prefix = prefix
        self.count = 0

    def _name(self):
        self.count += 1
        return "%s%d" % (self.prefix, self.count - 1)

    def _group(self, terms):
        # terms: list of (sign, var) with sign +-1
        key = tuple(sorted(terms))
        if len(terms) == 1 and terms[0][0] == 1:
            return terms[0][1]
        if key not in self.cache:
            self.cache[key] = self._name()
            self.sums.append((self.cache[key], list(terms)))
        return self.cache[key]

    @property
    def lines(self):
        """The sums with their common pairs (a + b or a - b, up to the sign of the whole)
        taken out, the most frequent first, then the lines that use them."""
        sums = {name: dict((v, sg) for sg, v in terms) for name, terms in self.sums}
        order = list(sums)
        count, tried = self.count, set()
        while self.fuse:
            pairs = {}
            for name in order:
                vs = sorted(sums[name])
                for i, u in enumerate(vs):
                    for v in vs[i + 1:]:
                        pairs.setdefault((u, v, sums[name][u] * sums[name][v]), []).append(name)
            best = max((q for q in pairs if q not in tried and len(pairs[q]) > 1),
                       key=lambda q: (len(pairs[q]), q), default=None)
            if best is None:
                break
            tried.add(best)
            u, v, rel = best
            new = next((n for n in pairs[best] if len(sums[n]) == 2 and sums[n][u] > 0), None)
            if new is None:
                new, count = "%s%d" % (self.prefix, count), count + 1
                sums[new] = {u: 1, v: rel}
                order.append(new)
            for name in pairs[best]:
                if name != new and new not in sums[name]:
                    sg = sums[name].pop(u)
                    del sums[name][v]
                    sums[name][new] = sg
        out, done = [], set()

        def emit(name):
            if name in done or name not in sums:
                return
            done.add(name)
            for v in sums[name]:
                emit(v)
            pos = [v for v, sg in sums[name].items() if sg > 0]
            neg = [v for v, sg in sums[name].items() if sg < 0]
            expr = " + ".join(pos) + "".join(" - %s" % v for v in neg) if pos else "-(" + " + ".join(neg) + ")"
            out.append("const C %s = %s;" % (name, expr))
        for name in order:
            emit(name)
        return out + self.late

    def combo(self, coeffs):
        """coeffs: list of (Fraction, var). Returns a C expression."""
        groups = {}
        for c, v in coeffs:
            if c == 0:
                continue
            a = abs(c)
            groups.setdefault(a, []).append((1 if c > 0 else -1, v))
        if not groups:
            return "C(0.0)"
        parts = []
        # with fuse the sum without a product first
        for a in sorted(groups, key=lambda x: (self.fuse and x != 1, x)):
            g = self._group(groups[a])
            parts.append(g if a == 1 else "%s*%s" % (_lit(a), g))
        return " + ".join(parts)


def _transform(builder, mat, invars, outvars, ksym, sig, rows_are_outputs=True):
    """Lines computing outvars = mat @ invars (f2m) using pair parity if available."""
    ns = len(mat)
    lines = []
    if ksym is not None and sig is not None:
        # pair sums/differences of the inputs
        reps = [k for k in range(ns) if k <= ksym[k]]
        P, D = {}, {}
        for k in reps:
            if ksym[k] == k:
                P[k] = invars[k]
            else:
                P[k] = builder._group([(1, invars[k]), (1, invars[ksym[k]])])
                D[k] = builder._group([(1, invars[k]), (-1, invars[ksym[k]])])
        for i in range(ns):
            coeffs = []
            for k in reps:
                c = mat[i][k]
                if c == 0:
                    continue
                if sig[i] > 0:
                    coeffs.append((c, P[k]))
                elif ksym[k] != k:
                    coeffs.append((c, D[k]))
            lines.append((outvars[i], builder.combo(coeffs)))
    else:
        for i in range(ns):
            lines.append((outvars[i], builder.combo([(mat[i][j], invars[j]) for j in range(ns)])))
    return lines


def _inverse_transform(builder, inv, mvars, fvars, ksym, sig, tag=""):
    """Lines computing fvars = inv @ mvars (entries of mvars that are None are zero);
    with parity f_k = E_k + O_k, f_ksym = E_k - O_k."""
    ns = len(inv)
    lines = []

    if ksym is not None and sig is not None:
        for k in range(ns):
            if k > ksym[k]:
                continue
            even = [(inv[k][i], mvars[i]) for i in range(ns) if sig[i] > 0 and mvars[i] is not None]
            odd = [(inv[k][i], mvars[i]) for i in range(ns) if sig[i] < 0 and mvars[i] is not None]
            if ksym[k] == k:
                lines.append((fvars[k], builder.combo(even)))
                continue
            e = "E%s%d" % (tag, k)
            o = "O%s%d" % (tag, k)
            builder.late.append("const C %s = %s;" % (e, builder.combo(even)))
            builder.late.append("const C %s = %s;" % (o, builder.combo(odd)))
            lines.append((fvars[k], "%s + %s" % (e, o)))
            lines.append((fvars[ksym[k]], "%s - %s" % (e, o)))
    else:
        for k in range(ns):
            lines.append((fvars[k], builder.combo([(inv[k][i], mvars[i]) for i in range(ns)
                                                   if mvars[i] is not None])))
    return lines


def _deviation_eq(expr, full, rest):
    """eq(c_ref + m') - eq(c_ref) with the constant cancelled symbolically."""
    e = sp.expand(sp.sympify(expr).xreplace(full) - sp.sympify(expr).xreplace(rest))
    zero = {s: 0 for s in full}
    if sp.simplify(e.xreplace(zero)) != 0:
        e = sp.cancel(sp.together(e))
    return e


def _collision_lines(spec: KernelSpec, with_sources: bool, fuse=True):
    """Full-value collision (FP64, as pylbm): sources, relax, sources on m0..m{ns-1}."""
    ns, nc = spec.ns, spec.nconsm
    out = []

    def sources():
        for idx, expr in spec.sources:
            out.append("m%d = m%d + half_dt * (%s);" % (idx, idx, _ccode(sp.sympify(expr), fuse)))

    if with_sources and spec.sources:
        sources()
    relaxed = [i for i in range(nc, ns) if spec.s[i] != 0]
    repl, red = sp.cse([spec.eq[i] for i in relaxed], symbols=sp.numbered_symbols("q_"),
                       optimizations="basic")
    for sym, e in repl:
        out.append("const C %s = %s;" % (sym, _ccode(e, fuse)))
    for i, e in zip(relaxed, red):
        out.append("m%d = one_minus[%d] * m%d + omega[%d] * (%s);" % (i, i, i, i, _ccode(e, fuse)))
    if with_sources and spec.sources:
        sources()
    return out


def _deviation_collision_lines(spec: KernelSpec, fuse):
    """Collision of the FP32-compute formats, in increments.

    The m_i are moments of d = f - w (w the rest populations of the reference
    state c_ref = (rho0, 0, ..., 0), rho0 = cref[0] at run time), so the
    conserved moments are c_ref + m_c and the target of a relaxed row is
    eq_i(c_ref + m_c) - eq_i(c_ref).  The kernel computes the change of every
    moment, dm_i = s_i (eq_i' - m_i) for relaxed rows and the source half
    steps for source rows, and applies fnew = d + M^-1 dm: equal in exact
    arithmetic to M^-1 (m + dm), but the rounding of the M^-1 coefficients
    now multiplies the small non-equilibrium change instead of the moments,
    and the rest state (dm = 0) is reproduced exactly.

    Returns (lines, names) with names[i] the C name of dm_i or None."""
    ns, nc = spec.ns, spec.nconsm
    msyms = spec.msyms
    crefs = [sp.Symbol("cr0")] + [sp.Integer(0)] * (nc - 1) if nc else []
    full = {msyms[i]: crefs[i] + msyms[i] for i in range(nc)}
    rest = {msyms[i]: crefs[i] for i in range(nc)}
    out = []
    names = [None] * ns
    src_rows = sorted({idx for idx, _ in spec.sources})
    for idx in src_rows:
        out.append("C dm%d = C(0.0);" % idx)
        names[idx] = "dm%d" % idx

    def sources():
        for idx, expr in spec.sources:
            e = sp.sympify(expr).xreplace(full)
            out.append("{ const C inc = half_dt * (%s); m%d += inc; dm%d += inc; }" % (_ccode(e, fuse), idx, idx))

    sources()
    relaxed = [i for i in range(nc, ns) if spec.s[i] != 0]
    eqs = [_deviation_eq(spec.eq[i], full, rest) for i in relaxed]
    repl, red = sp.cse(eqs, symbols=sp.numbered_symbols("q_"), optimizations="basic")
    for sym, e in repl:
        out.append("const C %s = %s;" % (sym, _ccode(e, fuse)))
    for i, e in zip(relaxed, red):
        if fuse:
            target = _ccode(sp.sympify(e) - msyms[i])
        else:
            target = "%s - m%d" % ("C(0.0)" if e == 0 else "(%s)" % _ccode(e, False), i)
        if names[i] is None:
            out.append("C dm%d = omega[%d] * (%s);" % (i, i, target))
            names[i] = "dm%d" % i
        else:
            out.append("{ const C inc = omega[%d] * (%s); dm%d += inc; m%d += inc; }" % (i, target, i, i))
            continue
        out.append("m%d += dm%d;" % (i, i))
    sources()
    return out, names


def _relative_collision_lines(spec: KernelSpec):
    """Collision of a relative-velocity scheme on m = M f (pylbm/algorithm/pull.py:38-59
    with base.py:255-263, 316-331, 366-368, 404-428), in full values:

    u = rel_vel(m_c); mr = T(u) m (the rows of Mu f = T(u) M f); the non-conserved
    rows take their relative values; [source dt/2]; relaxed rows
    m_i <- (1 - s_i) m_i + s_i (T(u) eq(m_c))_i; the conserved rows take their
    relative values mr_c (restore_conserved_moments); [source dt/2]; then
    ma = T(-u) m, whose M^-1 gives the new populations.

    Returns (lines, names) with names[i] the C name of ma_i."""
    ns, nc = spec.ns, spec.nconsm
    msyms = spec.msyms
    out = []
    for d, e in enumerate(spec.rel_vel):
        out.append("const C ru%d = %s;" % (d, _ccode(e, False)))
    Tu = [[sp.sympify(c) for c in r] for r in spec.Tu]
    Tmu = [[sp.sympify(c) for c in r] for r in spec.Tmu]

    def rows(mat, vec, which, prefix):
        exprs = [sum((mat[i][j] * vec[j] for j in range(ns) if mat[i][j] != 0), sp.Integer(0)) for i in which]
        repl, red = sp.cse(exprs, symbols=sp.numbered_symbols(prefix), optimizations="basic")
        lines = ["const C %s = %s;" % (sym, _ccode(e, False)) for sym, e in repl]
        return lines, red

    # relative moments of the pulled populations
    lines, red = rows(Tu, msyms, range(ns), "tr_")
    out += lines
    out += ["const C mr%d = %s;" % (i, _ccode(e, False)) for i, e in zip(range(ns), red)]
    out += ["m%d = mr%d;" % (i, i) for i in range(nc, ns)]

    def sources():
        for idx, expr in spec.sources:
            out.append("m%d = m%d + half_dt * (%s);" % (idx, idx, _ccode(sp.sympify(expr), False)))

    sources()
    relaxed = [i for i in range(nc, ns) if spec.s[i] != 0]
    eqv = [msyms[j] if j < nc else sp.sympify(spec.eq[j]) for j in range(ns)]
    lines, red = rows(Tu, eqv, relaxed, "te_")
    out += lines
    for i, e in zip(relaxed, red):
        out.append("m%d = one_minus[%d] * m%d + omega[%d] * (%s);" % (i, i, i, i, _ccode(e, False)))
    out += ["m%d = mr%d;" % (i, i) for i in range(nc)]
    sources()
    lines, red = rows(Tmu, msyms, range(ns), "ta_")
    out += lines
    out += ["const C ma%d = %s;" % (i, _ccode(e, False)) for i, e in zip(range(ns), red)]
    return out, ["ma%d" % i for i in range(ns)]


def _equilibrium_lines(spec: KernelSpec):
    ns, nc = spec.ns, spec.nconsm
    rows = list(range(nc, ns))
    repl, red = sp.cse([spec.eq[i] for i in rows], symbols=sp.numbered_symbols("q_"),
                       optimizations="basic")
    out = ["const C %s = %s;" % (s, _ccode(e)) for s, e in repl]
    for i, e in zip(rows, red):
        out.append("m%d = %s;" % (i, _ccode(e)))
    return out


# ------------------------------------------------------------------ template
_TEMPLATE = r"""// Generated by pylbm_amd.generator.hip for scheme %(hash)s -- do not edit.
// ns=%(ns)d nconsm=%(nc)d dim=%(dim)d pair-factored=%(paired)s
// Population stores may bypass the caches (stream_stores).
#ifndef LBM_NT_STORES
#define LBM_NT_STORES 1
#endif
#include "lbm_device.h"
#include <type_traits>

using namespace lbm;

#define NS %(ns)d
#define BBSUB_OK %(bbsub_ok)d  // the step can substitute fused bounce-back pulls
#define NCONSM %(nc)d
#define NCREF (NCONSM > 0 ? NCONSM : 1)
#define DIM %(dim)d
#define TB_UNIT_VELOCITIES %(unit_vel)d  // every velocity component in {-1, 0, 1}
#ifndef TB_THREADS
#define TB_THREADS 1024                // threads of a temporally blocked workgroup
#endif
#define TB_MAX_NT (DIM == 1 ? 64 : 16) // steps per temporally blocked launch, at most
#define TB_PLANE_1D 256                // cells of a 1D region, at most
#define TB_MASK %(bbsub_ok)d                    // folded links possible
#define TB_BATCH (sizeof(S) == 8 && DIM == 2 ? 1 : 2)   // cells a thread of a blocked workgroup loads at once
#define TB_LINKS 4                     // folded links a thread of a blocked workgroup holds
#define PAIR_OK %(pair_ok)d            // the two-step kernel is generated

namespace {

template <typename C>
struct StepArgs {
  int64_t src_off[NS];   // pull source offset of population k relative to the cell
  int64_t dst_off[NS];   // k * pop_stride
  int32_t nin[3];        // interior extents
  int32_t halo[3];
  int32_t n1, rs, lead, remap;     // rs: elements between consecutive rows; remap: XCD-aware order
  int32_t ends_first;              // planes from both ends to the middle
  int32_t nt;                      // population stores past the caches
  const uint32_t* bbmask;          // NULL or folded link directions per interior cell
  const uint32_t* bbtab_bits;      // NULL or the folded links with a sign / value table entry
  const uint32_t* bbtab_base;
  const uint32_t* bbtab_src;
  const C* bbtab_sign;
  const C* bbtab_rhs;
  const uint32_t* bbtab_rel;       // NULL or the table sources relative to the pulling cell
  const uint32_t* bbtab_src2;      // NULL or second sources (0xffffffff: a one-source entry)
  const C* bbtab_c2;
  const uint32_t* bbtab_rel2;
  C omega[NS], one_minus[NS], wshift[NS];
  C cref[NCREF];
  C half_dt, t;
  C xorg[3], dx;         // cell centre of reference axis d: xorg[d] + dx * (halo-inclusive index)
};

// Launch shape: LBM_BX threads along the contiguous axis x block_rows<S>() rows
// per workgroup (LBM_BY when set above 1), each thread updating LBM_MROWS
// consecutive rows of its column.
#ifndef LBM_BX
#define LBM_BX 256
#endif
#ifndef LBM_BY
#define LBM_BY 1
#endif
#ifndef LBM_MROWS
#define LBM_MROWS 1
#endif

// Cells per thread along the contiguous axis of the vector instantiation (vector
// loads / stores): 0 = by element size: 4 cells for the 4-byte formats (16 B per
// lane) and the 2-byte formats (8 B per lane, pulled rows at odd offsets assembled
// by vload_pull), 1 for FP64 (measured no gain on MI355X).
#ifndef LBM_VEC
#define LBM_VEC 0
#endif
#ifndef LBM_FORCE_I64
#define LBM_FORCE_I64 0
#endif
// whether the launch picks the vector instantiation by itself for the 2-byte formats
#ifndef LBM_VEC16_AUTO
#define LBM_VEC16_AUTO 0
#endif
// Rows of a fused-step workgroup: LBM_BY, or by default 2 for FP64 and 1 for the
// other formats (MI355X, 256^3 D3Q19: FP64 0.913 ms per step with 2 rows against
// 0.921 with 1; FP32 0.458 against 0.449)
template <typename S>
__host__ __device__ constexpr int block_rows() {
  return LBM_BY > 1 ? LBM_BY : (sizeof(S) == 8 ? 2 : 1);
}

// Waves per SIMD of a fused step.  FP64 in 3D, at least 4: source terms in X, Y, Z and t
// bring D3Q19 to 129 registers, one more than 4 waves have (200^3 432 us per step with 3, 421).
// Stores past the caches in 3D, 16 populations and more, where more waves stream slower: 2-byte
// formats and FP32 at most 5 (with 6, 200^3 FP16 takes 135 us instead of 129, 230 x 210 x 220 164
// instead of 158, 144^3 FP32 86.0 instead of 84.7; 6 populations stream faster with all 8, 200^3
// FP16 47 us instead of 58); FP32 with four cells per thread at most 2 (with 3, 200^3 240 us
// instead of 237, 230 x 210 x 220 313 instead of 307).
template <typename S, bool TABLE>
constexpr int least_waves() {
  return sizeof(S) == 8 && DIM == 3 && NS <= 19 && !TABLE ? 4 : 1;
}
template <typename S, int VEC, bool NT>
constexpr int most_waves() {
  if (DIM < 3 || NS < 16 || !NT) return 8;
  return sizeof(S) == 2 ? 5 : Codec<S>::kind == LBM_F32 ? (VEC > 1 ? 2 : 5) : 8;
}

template <typename S>
constexpr int vec_cells() {
  return LBM_VEC > 0 ? LBM_VEC : (sizeof(S) <= 4 ? 4 : 1);
}

// Workgroup order: consecutive workgroups are dealt round-robin to the 8 XCDs of
// MI355X.  With remap the linear workgroup index is renumbered so that each XCD
// takes a contiguous range of (mid, outer) rows, whose pulled neighbour rows then
// hit the same L2 (only when the count is a multiple of 8).  A run-time choice
// (lbm_params.xcd_remap; by default on for the halo path, off for the wrap path).
__device__ __forceinline__ void block_coords(unsigned& bx, unsigned& by, unsigned& bz, int remap) {
  bx = blockIdx.x;
  by = blockIdx.y;
  bz = blockIdx.z;
  if (remap) {
    const unsigned total = gridDim.x * gridDim.y * gridDim.z;
    if (total %% 8 == 0) {
      const unsigned lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
      const unsigned logical = (lin %% 8) * (total / 8) + lin / 8;
      bx = logical %% gridDim.x;
      by = (logical / gridDim.x) %% gridDim.y;
      bz = logical / (gridDim.x * gridDim.y);
    }
  }
}

// memory from an offset of an array on as a buffer: an address is its start, an offset in a
// scalar register and one in a vector register (32 bits each), without vector arithmetic
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* p, uint64_t offset) {
  return __builtin_amdgcn_make_buffer_rsrc((char*)const_cast<void*>(p) + offset, 0, 0xffffffffu, 0x00020000);
}
// non-temporal (aux bit 1) or not
template <typename S, bool NT>
__device__ __forceinline__ void buffer_store(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s, S x) {
  if constexpr (sizeof(S) == 8) {
    typedef uint32_t v2 __attribute__((ext_vector_type(2)));
    v2 b;
    __builtin_memcpy(&b, &x, 8);
    __builtin_amdgcn_raw_buffer_store_b64(b, r, v, s, NT ? 2 : 0);
  } else if constexpr (sizeof(S) == 4) {
    uint32_t b;
    __builtin_memcpy(&b, &x, 4);
    __builtin_amdgcn_raw_buffer_store_b32(b, r, v, s, NT ? 2 : 0);
  } else {
    uint16_t b;
    __builtin_memcpy(&b, &x, 2);
    __builtin_amdgcn_raw_buffer_store_b16(b, r, v, s, NT ? 2 : 0);
  }
}

// I: the element index type, int32_t when every index of the array fits it (the
// usual case: 32-bit offsets from a 64-bit base), int64_t for larger arrays.  NT: the
// population stores bypass the caches (stream_stores); a branch on it inside the kernel
// would be merged into one kind of store.  TABLE: folded links may have table entries; their
// batched loads take registers (D2Q9 FP64 48 -> 130) that boxes without a table need not pay.
template <typename S, bool FOLD, int VEC, typename I, bool NT, bool TABLE>
__global__ void __launch_bounds__(LBM_BX * block_rows<S>())
__attribute__((amdgpu_waves_per_eu(least_waves<S, TABLE>(), most_waves<S, VEC, NT>())))
fused_step(const S* __restrict__ f, S* __restrict__ fn, const StepArgs<typename Codec<S>::C> a) {
  using C = typename Codec<S>::C;
  // full-value arithmetic for FP64 (as pylbm), deviations from the rest state otherwise
  constexpr bool DEV = Codec<S>::kind != LBM_F64;
  unsigned bkx, bky, bkz;
  block_coords(bkx, bky, bkz, a.remap);
  const int i = (bkx * blockDim.x + threadIdx.x) * VEC;
  if (i >= a.nin[2]) return;
  // with table entries the planes go from both ends to the middle: inflow and outflow faces,
  // whose waves take several times as long, do not come last
  const int oo = TABLE && a.ends_first ? ((bkz & 1) ? a.nin[0] - 1 - (int)(bkz >> 1) : (int)(bkz >> 1)) : (int)bkz;
  const int mbase = (bky * blockDim.y + threadIdx.y) * LBM_MROWS;
  const C half_dt = a.half_dt;
  const C tt = a.t;
  (void)half_dt; (void)tt;
  const C* one_minus = a.one_minus;
  const C* omega = a.omega;
  const C* cref = a.cref;
  (void)cref;
#pragma unroll
  for (int r = 0; r < LBM_MROWS; ++r) {
  const int mm = mbase + r;
  if (mm >= a.nin[1]) return;
  const int o = oo + a.halo[0], m = mm + a.halo[1], ii = i + a.halo[2];
  const I cell = ((I)o * a.n1 + m) * a.rs + a.lead + ii;
%(loads)s
%(bbsub)s
%(gdecl)s
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
%(coords)s
%(decode)s
%(collide)s
  }
%(vstores)s
  }
}

%(tb_kernel)stemplate <typename S>
__global__ void __launch_bounds__(256)
f2m_kernel(const S* __restrict__ f, lbm_layout fl, double* __restrict__ mo, lbm_layout ml,
           const StepArgs<double> a) {
#pragma clang fp contract(on)
  using C = double;
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= fl.n[2]) return;
  const int64_t m_ = blockIdx.y, o_ = blockIdx.z;
  const int64_t cf = cell_offset(fl, o_, m_, i);
  const int64_t cm = cell_offset(ml, o_, m_, i);
%(f2m_loads)s
%(f2m_full)s
%(f2m_stores)s
}

template <typename S>
__global__ void __launch_bounds__(256)
m2f_kernel(const double* __restrict__ mi, lbm_layout ml, S* __restrict__ f, lbm_layout fl,
           const StepArgs<double> a) {
#pragma clang fp contract(on)
  using C = double;
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= fl.n[2]) return;
  const int64_t m_ = blockIdx.y, o_ = blockIdx.z;
  const int64_t cf = cell_offset(fl, o_, m_, i);
  const int64_t cm = cell_offset(ml, o_, m_, i);
%(m2f_loads)s
%(m2f_full)s
%(m2f_stores)s
}

__global__ void __launch_bounds__(256)
equilibrium_kernel(double* __restrict__ mo, lbm_layout ml) {
#pragma clang fp contract(on)
  using C = double;
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= ml.n[2]) return;
  const int64_t m_ = blockIdx.y, o_ = blockIdx.z;
  const int64_t cm = cell_offset(ml, o_, m_, i);
%(eq_loads)s
%(eq_body)s
%(eq_stores)s
}

// pylbm's split routines, generated from the same spec: transport
// (pylbm/algorithm/base.py:273-296: fnew[k, x] = f[k, x - v_k] on the interior, a
// copy of the stored words), relaxation (404-437: m_i <- (1 - s_i) m_i + s_i eq_i
// on the whole halo-inclusive domain, FP64 moments) and source_term (439-504 with
// algorithm/ode.py:11-16: one explicit Euler half step m_c <- m_c + dt/2 S(m) on
// the interior, FP64 moments)
template <typename S>
__global__ void __launch_bounds__(256)
transport_kernel(const S* __restrict__ f, S* __restrict__ fn, const StepArgs<typename Codec<S>::C> a) {
  using B = typename Bits<S>::T;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.nin[2]) return;
  const int64_t cell = ((int64_t)(blockIdx.z + a.halo[0]) * a.n1 + blockIdx.y + a.halo[1]) * a.rs + a.lead + i +
                       a.halo[2];
  const B* fb = reinterpret_cast<const B*>(f);
  B* gb = reinterpret_cast<B*>(fn);
#pragma unroll
  for (int k = 0; k < NS; ++k) gb[a.dst_off[k] + cell] = fb[a.src_off[k] + cell];
}

__global__ void __launch_bounds__(256)
relaxation_kernel(double* __restrict__ mo, lbm_layout ml, const StepArgs<double> a) {
#pragma clang fp contract(on)
  using C = double;
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= ml.n[2]) return;
  const int64_t m_ = blockIdx.y, o_ = blockIdx.z;
  const int64_t cm = cell_offset(ml, o_, m_, i);
  const C* one_minus = a.one_minus;
  const C* omega = a.omega;
  (void)one_minus; (void)omega;
%(rx_loads)s
%(rx_body)s
%(rx_stores)s
}

__global__ void __launch_bounds__(256)
source_term_kernel(double* __restrict__ mo, lbm_layout ml, const StepArgs<double> a) {
#pragma clang fp contract(on)
  using C = double;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.nin[2]) return;
  const int o = (int)blockIdx.z + a.halo[0], m = (int)blockIdx.y + a.halo[1], ii = i + a.halo[2];
  (void)o; (void)m;
  constexpr int j = 0;
  (void)j;
  const int64_t cm = cell_offset(ml, o, m, ii);
  const C half_dt = a.half_dt;
  const C tt = a.t;
  (void)half_dt; (void)tt;
%(st_coords)s
%(st_loads)s
%(st_body)s
%(st_stores)s
}

// A value the compiler must treat as opaque: an equilibrium moment used as if it
// had been stored and loaded again, so that none of its products is contracted
// into an FMA of m2f's sums (which would round differently from the two-kernel path).
__device__ __forceinline__ double stored_moment(double x) {
  asm("" : "+v"(x));
  return x;
}

// equilibrium from the conserved moments followed by m2f, the moments kept in
// registers: the same expressions as equilibrium_kernel then m2f_kernel, so the
// same populations (the non-conserved rows of mo are not written)
template <typename S>
__global__ void __launch_bounds__(256)
eq_m2f_kernel(const double* __restrict__ mo, lbm_layout ml, S* __restrict__ f, lbm_layout fl,
              const StepArgs<double> a) {
#pragma clang fp contract(on)
  using C = double;
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= fl.n[2]) return;
  const int64_t m_ = blockIdx.y, o_ = blockIdx.z;
  const int64_t cf = cell_offset(fl, o_, m_, i);
  const int64_t cm = cell_offset(ml, o_, m_, i);
%(eqm2f_loads)s
%(eq_body)s
%(eqm2f_opaque)s
%(m2f_full)s
%(m2f_stores)s
}

// Population stores bypass the caches, unless the interior cells of both arrays hold 24 MiB
// to a limit: the next step then finds them in the 256 MB Infinity Cache.  The padding of the
// rows is not stored, so it does not count.  us per step past / into the caches:
// below 24 MiB: 64^3 D3Q19 FP16 (19 MiB) 7.1 / 7.8, 40^3 FP64 (19) 7.6 / 8.1, 512^2 D2Q9 FP32
// (18) 6.4 / 6.7; above: 56^3 FP32 (25) 8.3 / 8.1, 72^3 FP16 (27) 11.5 / 10.6, 96^3 FP32 (128) 26.1 / 23.0.
// Single steps to 306 MiB: 96^3 FP64 (257) 49.1 / 45.4, 128^3 FP32 (304) 61.0 / 53.4, 136^3
// FP32 (365) 75 / 105, 112^3 FP64 (407) 75.9 / 83.4.  2-byte formats in 3D to 176 MiB: 128^3 FP16
// (152) 29.2 / 25.4, D3Q15 160^3 (235) 47 / 51, 160^3 (297) 61 / 68.  Pairs to 256 MiB: 112^3 FP32
// (204) 38.0 / 32.6, 120^3 FP32 (251) 43.2 / 40.3, 96^3 FP64 (257) 35.3 / 37.0, D3Q6 180^3 FP32
// (267) 38.5 / 40.4.
static int stream_stores(const lbm_layout* L, int64_t most) {
  int64_t bytes = 2 * (int64_t)L->ns * storage_elem_size(L->storage);
  for (int d = 0; d < 3; ++d) bytes *= L->n[d] - 2 * L->halo[d];
  return bytes < (int64_t)24 << 20 || bytes > most << 20;
}

template <typename C>
static int make_args(const lbm_layout* L, const lbm_params* p, StepArgs<C>* a) {
  int rc = check_layout(L);
  if (rc) return rc;
  LBM_REQUIRE(L->ns == NS, "layout has ns=%%d, module was generated for %%d", L->ns, NS);
  static const int hv[NS][3] = {%(vel)s};
  for (int k = 0; k < NS; ++k) {
    a->dst_off[k] = k * L->pop_stride;
    a->src_off[k] = k * L->pop_stride - ((int64_t)hv[k][0] * L->n[1] + hv[k][1]) * L->row_stride - hv[k][2];
  }
  for (int d = 0; d < 3; ++d) {
    a->nin[d] = (int32_t)(L->n[d] - 2 * L->halo[d]);
    a->halo[d] = L->halo[d];
  }
  a->n1 = (int32_t)L->n[1];
  a->rs = (int32_t)L->row_stride;
  a->lead = (int32_t)L->lead;
  a->remap = 0;
  a->ends_first = 0;
  a->nt = stream_stores(L, storage_elem_size(L->storage) == 2 && DIM == 3 ? 176 : 306);
  for (int k = 0; k < NS; ++k) {
    a->omega[k] = p ? (C)p->omega[k] : (C)0;
    a->one_minus[k] = p ? (C)p->one_minus[k] : (C)1;
    a->wshift[k] = p ? (C)p->wshift[k] : (C)0;
  }
  for (int c = 0; c < NCREF; ++c) a->cref[c] = p ? (C)p->cref[c] : (C)0;
  a->half_dt = p ? (C)(0.5 * p->dt) : (C)0;
  a->t = p ? (C)p->t : (C)0;
  for (int d = 0; d < 3; ++d) a->xorg[d] = p ? (C)p->origin[d] : (C)0;
  a->dx = p ? (C)p->dx : (C)0;
  a->bbmask = p ? p->bbmask : nullptr;
  a->bbtab_bits = p ? p->bbtab_bits : nullptr;
  a->bbtab_base = p ? p->bbtab_base : nullptr;
  a->bbtab_src = p ? p->bbtab_src : nullptr;
  a->bbtab_sign = p ? (const C*)p->bbtab_sign : nullptr;
  a->bbtab_rhs = p ? (const C*)p->bbtab_rhs : nullptr;
  a->bbtab_rel = p ? p->bbtab_rel : nullptr;
  a->bbtab_src2 = p ? p->bbtab_src2 : nullptr;
  a->bbtab_c2 = p ? (const C*)p->bbtab_c2 : nullptr;
  a->bbtab_rel2 = p ? p->bbtab_rel2 : nullptr;
  LBM_REQUIRE(a->bbmask == nullptr || BBSUB_OK, "this stencil has no symmetric pairs: no fused bounce-back");
  return 0;
}

static unsigned block_x(int64_t n) {
  return n >= 256 ? 256u : (n >= 128 ? 128u : 64u);
}

template <typename S, bool FOLD, bool TABLE>
static void fused_launch(const S* f, S* fn, const StepArgs<typename Codec<S>::C>& a, bool narrow, int vec, dim3 grid,
                         dim3 block, hipStream_t s) {
  constexpr int V = vec_cells<S>();
  const auto go = [&](auto kernel) { kernel<<<grid, block, 0, s>>>(f, fn, a); };
  if constexpr (V > 1 && !TABLE) {
    if (vec == V) {
      if (narrow) go(fused_step<S, FOLD, V, int32_t, true, false>);
      else go(fused_step<S, FOLD, V, int64_t, true, false>);
      return;
    }
  }
  if (!narrow) go(fused_step<S, FOLD, 1, int64_t, true, TABLE>);
  else if (a.nt) go(fused_step<S, FOLD, 1, int32_t, true, TABLE>);
  else go(fused_step<S, FOLD, 1, int32_t, false, TABLE>);
}

template <typename S>
static int step_launch(const void* f, void* fn, const lbm_layout* L, const lbm_params* p, int fold,
                       hipStream_t s) {
  using C = typename Codec<S>::C;
  StepArgs<C> a;
  int rc = make_args<C>(L, p, &a);
  if (rc) return rc;
  constexpr int V = vec_cells<S>();
  // V cells per thread only where that still leaves >= 2^20 threads: small grids
  // (a 512^2 plane) need the waves of one cell per thread to hide memory latency.
  // Only the wrap path without folded links takes V cells: with a mask word per
  // cell the per-cell mask branches of a V-cell thread cost more than the wider
  // loads save, and the halo path's pulls straddle more cache lines (MI355X, 512 x
  // 256 x 256 D3Q19 sphere packing FP32: 0.90 ms per step with one cell per thread,
  // 0.93 with 2, 0.98 with 4; 256^3 halo path FP32 with its ghost fill: 0.514 ms
  // with one, 0.534 with 4).
  const int64_t cells = (int64_t)a.nin[0] * a.nin[1] * a.nin[2];
  const int want = p ? p->vec_cells : 0;
  LBM_REQUIRE(want == 0 || want == 1 || (want == V && a.nin[2] %% V == 0),
              "vec_cells %%d not available (%%d cells per thread, contiguous extent %%d)", want, V, a.nin[2]);
  // Stores into the caches go one cell per thread (180^3 D3Q6 FP32 46 us per step, 53 with 4
  // past them).
  const bool auto_vec = (sizeof(S) != 2 || LBM_VEC16_AUTO) && fold && a.bbmask == nullptr && a.nt;
  // cells with table entries are updated one per thread
  const int vec = a.bbtab_bits ? 1 : want ? want : ((auto_vec && a.nin[2] %% V == 0 && cells / V >= ((int64_t)1 << 20)) ? V : 1);
  a.remap = (p && p->xcd_remap >= 0) ? (p->xcd_remap != 0) : !fold;
  a.ends_first = fold && a.bbtab_bits && !a.remap;
  const int threads = a.nin[2] / vec;
  unsigned bx = LBM_BX;
  while (bx > 64 && (int)(bx / 2) >= threads) bx /= 2;
  const unsigned rows = block_rows<S>() * LBM_MROWS;
  dim3 block(bx, block_rows<S>());
  dim3 grid((unsigned)((threads + bx - 1) / bx), (unsigned)((a.nin[1] + rows - 1) / rows),
            (unsigned)a.nin[0]);
  if (fold) {
    for (int d = 0; d < 3; ++d)
      LBM_REQUIRE(a.nin[d] >= a.halo[d], "periodic fold needs extents >= halo");
  }
  const bool narrow = layout_fits_int32(*L) && !LBM_FORCE_I64;
  const auto go = [&](auto folded, auto table) {
    fused_launch<S, decltype(folded)::value, decltype(table)::value>((const S*)f, (S*)fn, a, narrow, vec, grid, block, s);
  };
  using T = std::integral_constant<bool, BBSUB_OK>;
  if (fold) a.bbtab_bits ? go(std::true_type{}, T{}) : go(std::true_type{}, std::false_type{});
  else a.bbtab_bits ? go(std::false_type{}, T{}) : go(std::false_type{}, std::false_type{});
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

template <typename S>
static int f2m_launch(const void* f, const lbm_layout* fl, double* mo, const lbm_layout* ml,
                      const lbm_params* p, hipStream_t s) {
  StepArgs<double> a;
  int rc = make_args<double>(fl, p, &a);
  if (rc) return rc;
  const unsigned bx = block_x(fl->n[2]);
  dim3 grid((unsigned)((fl->n[2] + bx - 1) / bx), (unsigned)fl->n[1], (unsigned)fl->n[0]);
  f2m_kernel<S><<<grid, bx, 0, s>>>((const S*)f, *fl, mo, *ml, a);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

template <typename S>
static int m2f_launch(const double* mi, const lbm_layout* ml, void* f, const lbm_layout* fl,
                      const lbm_params* p, hipStream_t s) {
  StepArgs<double> a;
  int rc = make_args<double>(fl, p, &a);
  if (rc) return rc;
  const unsigned bx = block_x(fl->n[2]);
  dim3 grid((unsigned)((fl->n[2] + bx - 1) / bx), (unsigned)fl->n[1], (unsigned)fl->n[0]);
  m2f_kernel<S><<<grid, bx, 0, s>>>(mi, *ml, (S*)f, *fl, a);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

template <typename S>
static int transport_launch(const void* f, void* fn, const lbm_layout* fl, const lbm_params* p, hipStream_t s) {
  StepArgs<typename Codec<S>::C> a;
  int rc = make_args<typename Codec<S>::C>(fl, p, &a);
  if (rc) return rc;
  const unsigned bx = block_x(a.nin[2]);
  dim3 grid((unsigned)((a.nin[2] + bx - 1) / bx), (unsigned)a.nin[1], (unsigned)a.nin[0]);
  transport_kernel<S><<<grid, bx, 0, s>>>((const S*)f, (S*)fn, a);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

template <typename S>
static int eq_m2f_launch(const double* mi, const lbm_layout* ml, void* f, const lbm_layout* fl,
                         const lbm_params* p, hipStream_t s) {
  StepArgs<double> a;
  int rc = make_args<double>(fl, p, &a);
  if (rc) return rc;
  const unsigned bx = block_x(fl->n[2]);
  dim3 grid((unsigned)((fl->n[2] + bx - 1) / bx), (unsigned)fl->n[1], (unsigned)fl->n[0]);
  eq_m2f_kernel<S><<<grid, bx, 0, s>>>(mi, *ml, (S*)f, *fl, a);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

%(tb_launch)sstatic int same_extents(const lbm_layout* a, const lbm_layout* b) {
  LBM_REQUIRE(a && b, "layout is NULL");
  LBM_REQUIRE(b->storage == LBM_F64, "moment layout must be FP64");
  for (int d = 0; d < 3; ++d)
    LBM_REQUIRE(a->n[d] == b->n[d], "moment / population extents differ on axis %%d", d);
  return check_layout(b);
}

}  // namespace

extern "C" {

int lbm_gen_info(int32_t* ns, int32_t* nconsm, int32_t* dim) {
  *ns = NS;
  *nconsm = NCONSM;
  *dim = DIM;
  return 0;
}

int lbm_gen_step(const void* d_f, void* d_fnew, const lbm_layout* layout, const lbm_params* params,
                 int periodic_fold, void* stream) {
  LBM_REQUIRE(layout, "layout is NULL");
  hipStream_t s = (hipStream_t)stream;
  LBM_DISPATCH_STORAGE(layout->storage, step_launch, d_f, d_fnew, layout, params, periodic_fold, s);
}

int lbm_gen_f2m(const void* d_f, const lbm_layout* fl, double* d_m, const lbm_layout* ml,
                const lbm_params* params, void* stream) {
  int rc = same_extents(fl, ml);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  LBM_DISPATCH_STORAGE(fl->storage, f2m_launch, d_f, fl, d_m, ml, params, s);
}

int lbm_gen_m2f(const double* d_m, const lbm_layout* ml, void* d_f, const lbm_layout* fl,
                const lbm_params* params, void* stream) {
  int rc = same_extents(fl, ml);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  LBM_DISPATCH_STORAGE(fl->storage, m2f_launch, d_m, ml, d_f, fl, params, s);
}

int lbm_gen_eq_m2f(const double* d_m, const lbm_layout* ml, void* d_f, const lbm_layout* fl,
                   const lbm_params* params, void* stream) {
  int rc = same_extents(fl, ml);
  if (rc) return rc;
  LBM_REQUIRE(ml->storage == LBM_F64 && ml->ns == NS, "eq_m2f needs FP64 moments of ns=%%d", NS);
  hipStream_t s = (hipStream_t)stream;
  LBM_DISPATCH_STORAGE(fl->storage, eq_m2f_launch, d_m, ml, d_f, fl, params, s);
}

int lbm_gen_equilibrium(double* d_m, const lbm_layout* ml, void* stream) {
  int rc = check_layout(ml);
  if (rc) return rc;
  LBM_REQUIRE(ml->storage == LBM_F64 && ml->ns == NS, "equilibrium needs FP64 moments of ns=%%d", NS);
  const unsigned bx = block_x(ml->n[2]);
  dim3 grid((unsigned)((ml->n[2] + bx - 1) / bx), (unsigned)ml->n[1], (unsigned)ml->n[0]);
  equilibrium_kernel<<<grid, bx, 0, (hipStream_t)stream>>>(d_m, *ml);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

int lbm_gen_transport(const void* d_f, void* d_fnew, const lbm_layout* fl, const lbm_params* params,
                      void* stream) {
  LBM_REQUIRE(d_f != d_fnew, "transport needs distinct source and destination arrays");
  hipStream_t s = (hipStream_t)stream;
  LBM_DISPATCH_STORAGE(fl ? fl->storage : -1, transport_launch, d_f, d_fnew, fl, params, s);
}

int lbm_gen_relaxation(double* d_m, const lbm_layout* ml, const lbm_params* params, void* stream) {
  LBM_REQUIRE(params != nullptr, "NULL params");
  StepArgs<double> a;
  int rc = make_args<double>(ml, params, &a);
  if (rc) return rc;
  LBM_REQUIRE(ml->storage == LBM_F64, "relaxation needs FP64 moments");
  const unsigned bx = block_x(ml->n[2]);
  dim3 grid((unsigned)((ml->n[2] + bx - 1) / bx), (unsigned)ml->n[1], (unsigned)ml->n[0]);
  relaxation_kernel<<<grid, bx, 0, (hipStream_t)stream>>>(d_m, *ml, a);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

int lbm_gen_source_term(double* d_m, const lbm_layout* ml, const lbm_params* params, void* stream) {
  LBM_REQUIRE(params != nullptr, "NULL params");
  StepArgs<double> a;
  int rc = make_args<double>(ml, params, &a);
  if (rc) return rc;
  LBM_REQUIRE(ml->storage == LBM_F64, "source_term needs FP64 moments");
  const unsigned bx = block_x(a.nin[2]);
  dim3 grid((unsigned)((a.nin[2] + bx - 1) / bx), (unsigned)a.nin[1], (unsigned)a.nin[0]);
  source_term_kernel<<<grid, bx, 0, (hipStream_t)stream>>>(d_m, *ml, a);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

int lbm_gen_run_blocked(void* d_f, void* d_fnew, const lbm_layout* layout, lbm_params* params,
                        int64_t nsteps, int steps_per_launch, int tile_m, int tile_i, int* parity,
                        void* stream) {
  LBM_REQUIRE(params && layout && parity, "NULL argument");
  LBM_REQUIRE(DIM <= 2, "temporal blocking is generated for 1D and 2D schemes only (this one is %%dD)", DIM);
  LBM_REQUIRE(TB_UNIT_VELOCITIES, "temporal blocking needs velocity components in {-1, 0, 1}");
  LBM_REQUIRE(steps_per_launch >= 1 && steps_per_launch <= TB_MAX_NT, "steps per launch out of [1, %%d]",
              TB_MAX_NT);
  LBM_REQUIRE(tile_m >= 1 && tile_i >= 1, "tile sizes must be positive");
  LBM_REQUIRE(params->bbtab_bits == nullptr || params->bbtab_rel != nullptr,
              "folded links with table entries need their relative sources (bbtab_rel)");
  LBM_REQUIRE(params->bbtab_src2 == nullptr || params->bbtab_rel2 != nullptr,
              "folded interpolated links need their relative second sources (bbtab_rel2)");
  hipStream_t s = (hipStream_t)stream;
  void* a = d_f;
  void* b = d_fnew;
  // nsteps in launches of at most steps_per_launch steps, as even as they come: 200
  // steps at most 6 at a time are 32 launches of 6 and 2 of 4, not 33 and two steps
  int64_t launches = (nsteps + steps_per_launch - 1) / steps_per_launch;
  if (!params->launch_parity) launches += (nsteps - launches) & 1;
  for (int64_t it = 0; it < launches; ++it) {
    const int nt = (int)(nsteps * (it + 1) / launches - nsteps * it / launches);
    int rc = 0;
    if (nt > 1) {
      LBM_DISPATCH_BLOCKED(layout->storage, tb_launch, a, b, layout, params, nt, tile_m, tile_i, s, rc);
    } else {
      rc = lbm_gen_step(a, b, layout, params, 1, stream);
      params->t += params->dt;
    }
    if (rc) return rc;
    void* tmp = a;
    a = b;
    b = tmp;
  }
  *parity = (int)(launches & 1);
  return 0;
}

int lbm_gen_run(void* d_f, void* d_fnew, const lbm_layout* layout, const lbm_velocities* vel,
                lbm_params* params, const lbm_link_set* links, int nmeth, int64_t nsteps,
                int ghost, int periodic_fold, int* parity, void* stream) {
  LBM_REQUIRE(params && layout && parity, "NULL argument");
  LBM_REQUIRE(!(periodic_fold && nmeth > 0), "periodic fold is only valid without link lists");
  void* a = d_f;
  void* b = d_fnew;
  int64_t launches = 0;
#if PAIR_OK
  // an even number of pairs leaves the result where single steps would have
  const int64_t paired = !periodic_fold ? 0 : params->launch_parity ? nsteps / 2 * 2 : nsteps / 4 * 4;
#endif
  for (int64_t it = 0; it < nsteps; ++it, ++launches) {
    int rc = 0;
#if PAIR_OK
    if (it < paired) {
      bool done;
      rc = pair_any(a, b, layout, params, &done, (hipStream_t)stream);
      if (rc) return rc;
      if (done) {
        ++it;
        void* tmp = a;
        a = b;
        b = tmp;
        continue;
      }
    }
#endif
    if (ghost == 1) rc = lbm_ghost_fill(a, layout, vel, stream);
    else if (ghost == 2) rc = lbm_ghost_fill_all(a, layout, vel, stream);
    if (rc) return rc;
    if (nmeth > 0) rc = lbm_links_apply_sets(a, layout, links, nmeth, stream);
    if (rc) return rc;
    rc = lbm_gen_step(a, b, layout, params, periodic_fold, stream);
    if (rc) return rc;
    void* tmp = a;
    a = b;
    b = tmp;
    params->t += params->dt;
  }
  *parity = (int)(launches & 1);
  return 0;
}

}  // extern "C"
"""


_TB_KERNEL = r"""// ------------------------------------------------ temporally blocked steps (2D)
// One workgroup advances a tm x ti tile of the interior (mid x inner axes) by nt
// steps in LDS: it loads the (tm + 2 nt) x (ti + 2 nt) region around the tile
// through the periodic wrap of the interior (valid where the wrap path is: a
// periodic box, or every link list folded into the mask / table), then for
// s = 1 .. nt computes the cells of the region shrunk by s from the values of
// step s - 1 with the per-cell arithmetic of fused_step (the same generated
// lines, so the same bits), and finally stores the tile.
//
// Folded links.  The link of population k at cell x gives the value that x pulls
// from (k, x - v_k), and no other cell pulls that slot, so a workgroup applies its
// links as pylbm's lists do: before each step every link's value is written into its
// slot of the LDS region, and the cells then pull without looking at a mask.  The
// load phase collects the region's links in a list (an LDS counter), one thread takes
// TB_LINKS of them at most and holds their slots, coefficients and values in
// registers for the whole launch; a step reads all sources, waits, and writes all
// slots (a slot may be another link's source where the region wraps around a small
// box).  Reading each table entry from memory in its cell, every step, one direction
// after the other, made the launch as slow as the tile with most of them (per step,
// entries in the cells / in the list: 901 x 219 channel around a cylinder,
// interpolated walls, FP32 deviations 5.8 / 3.4 us; with plain walls, 1024 x 256 FP32
// 3.8 / 3.4 us; 5000-cell 1D shock tube FP64 1.4 / 0.65 us).
// A region with more links than the list holds takes the mask, table bits and first
// entries of its cells into LDS and substitutes link by link in the cell.
template <typename C>
struct TbArgs {
  int32_t nt, tm, ti, tiles_i;
  uint32_t inv_ti, inv[TB_MAX_NT + 1];   // reciprocals of ti and of the row length after each step
  C times[TB_MAX_NT];   // t of each step (the host's sequence of t += dt)
};

// x in [-n, 3n) -> x mod n, without a division (tile regions reach at most nt < n
// cells before the interior and less than 2n + nt after its start)
__device__ __forceinline__ int wrap_near(int x, int n) {
  x += (x < 0) ? n : 0;
  x -= (x >= n) ? n : 0;
  x -= (x >= n) ? n : 0;
  return x;
}

// c / w for 0 <= c, w < 2^16 with inv = reciprocal(w): a 32-bit division is some 35
// instructions, and every thread needs one per step to find its cells
inline uint32_t reciprocal(int w) { return w > 1 ? (uint32_t)(((uint64_t)1 << 32) / w + 1) : 0u; }
__device__ __forceinline__ int divide(int c, uint32_t inv) {
  return inv ? (int)__umulhi((unsigned)c, inv) : c;
}

// Population planes of the region lie TB_PLANE<S> cells apart: a compile-time
// stride, so that the plane offsets of the pulls and stores become immediates of
// the LDS instructions.  It is the most cells the two copies of the populations
// plus the mask / table words fit in 160 KiB with, and keeps the last plane within
// the 16-bit immediate offset.
// With HALF a workgroup takes half the LDS and two share a CU: one loads or stores
// while the other computes.
template <typename S, bool HALF>
__host__ __device__ constexpr int tb_plane() {
  if (DIM == 1) return TB_PLANE_1D;
  constexpr int a = ((HALF ? 80 : 160) * 1024) / (2 * NS * (int)sizeof(S) + 12);
  constexpr int b = NS > 1 ? 65528 / ((NS - 1) * (int)sizeof(S)) : a;
  return a < b ? a : b;
}

template <typename S, bool HALF>
__global__ void __launch_bounds__(TB_THREADS)
tb_step(const S* __restrict__ f, S* __restrict__ fn, const StepArgs<typename Codec<S>::C> a,
        const TbArgs<typename Codec<S>::C> t) {
  using C = typename Codec<S>::C;
  constexpr bool DEV = Codec<S>::kind != LBM_F64;
  extern __shared__ uint4 tb_smem[];
  constexpr int MH = DIM == 2;   // the mid axis has a halo (a 1D region is one row)
  const int RW = t.tm + 2 * t.nt * MH, RI = t.ti + 2 * t.nt, RN = RW * RI;
  constexpr int RC = tb_plane<S, HALF>();   // plane stride (cells), RN <= RC
  S* cur = reinterpret_cast<S*>(tb_smem);
  S* nxt = cur + NS * RC;
  // the link list lives in nxt until the first step; dense regions keep their mask
  // words and, with table links, every cell's table bits and first entry after it
  constexpr int LIST_AT = (NS * RC * (int)sizeof(S) + 31) / 16 * 16;   // bytes, counter 16 before
  constexpr int LIST_FIT = (2 * NS * RC * (int)sizeof(S) - LIST_AT) / 8;
  int* nlinks = reinterpret_cast<int*>(reinterpret_cast<char*>(tb_smem) + LIST_AT - 16);
  uint2* links = reinterpret_cast<uint2*>(reinterpret_cast<char*>(tb_smem) + LIST_AT);
  const bool masked = TB_MASK && a.bbmask;
  const int cap = min(LIST_FIT, TB_LINKS * (int)blockDim.x);
  (void)nlinks; (void)links; (void)cap;
  if (masked) {
    if (threadIdx.x == 0) *nlinks = 0;
    __syncthreads();
  }
  uint32_t* msk = reinterpret_cast<uint32_t*>(cur + 2 * NS * RC);
  uint32_t* tbits = msk + RN;
  uint32_t* tbase_l = tbits + RN;
  const bool table = TB_MASK && a.bbmask && a.bbtab_bits;
  (void)msk; (void)tbits; (void)tbase_l; (void)table;
  const int m0 = (int)(blockIdx.x / t.tiles_i) * t.tm - t.nt * MH;
  const int i0 = (int)(blockIdx.x %% t.tiles_i) * t.ti - t.nt;
  const C half_dt = a.half_dt;
  (void)half_dt;
  const C* one_minus = a.one_minus;
  const C* omega = a.omega;
  const C* cref = a.cref;
  (void)cref;
  // TB_BATCH cells per thread in flight: all their loads are issued before the first
  // is written to LDS (2-byte and 4-byte formats without links 1 to 3 %% faster than one at a
  // time; FP64 in 2D 2 %% slower: 1000^2 D2Q9 + D2Q5 35.7 us per step with 2, 35.1 with 1)
  for (int c0 = threadIdx.x; c0 < RN; c0 += TB_BATCH * blockDim.x) {
    S v[TB_BATCH][NS];
    uint32_t bits_[TB_BATCH];
#pragma unroll
    for (int b = 0; b < TB_BATCH; ++b) {
      const int c = c0 + b * (int)blockDim.x;
      bits_[b] = 0;
      if (c < RN) {
        const int lr = divide(c, t.inv[0]);
        const int gm = wrap_near(m0 + lr, a.nin[1]), gi = wrap_near(i0 + c - lr * RI, a.nin[2]);
        const int64_t src = (int64_t)(a.halo[0] * a.n1 + gm + a.halo[1]) * a.rs + a.lead + gi + a.halo[2];
%(tb_mask)s
#pragma unroll
        for (int k = 0; k < NS; ++k) v[b][k] = f[a.dst_off[k] + src];
      }
    }
#pragma unroll
    for (int b = 0; b < TB_BATCH; ++b) {
      const int c = c0 + b * (int)blockDim.x;
      if (c < RN) {
#pragma unroll
        for (int k = 0; k < NS; ++k) cur[k * RC + c] = v[b][k];
      }
%(tb_collect)s
    }
  }
  __syncthreads();
%(tb_entries)s
  for (int s = 1; s <= t.nt; ++s) {
%(tb_apply)s
    const C tt = t.times[s - 1];
    (void)tt;
    const int WC = RI - 2 * s, HC = RW - 2 * s * MH;
    // the cells of the shrunk region in row-major order, blockDim.x apart: the
    // (row, column) of the next one follow by adding (dq, dr) with a carry, and its
    // region index by adding dl, plus dc on a carry (no multiply per cell)
    const int dq = divide((int)blockDim.x, t.inv[s]), dr = (int)blockDim.x - dq * WC;
    int rr = divide((int)threadIdx.x, t.inv[s]), qq = (int)threadIdx.x - rr * WC;
    const int dl = dq * RI + dr, dc = RI - WC;
    int lnext = (s * MH + rr) * RI + s + qq;
    for (int c = threadIdx.x; c < WC * HC; c += blockDim.x) {
      const int lr = s * MH + rr, lc = s + qq;
      const int lcell = lnext;
      qq += dr;
      rr += dq;
      lnext += dl;
      if (qq >= WC) {
        qq -= WC;
        ++rr;
        lnext += dc;
      }
      const int gm = wrap_near(m0 + lr, a.nin[1]), gi = wrap_near(i0 + lc, a.nin[2]);
      const int o = a.halo[0], m = gm + a.halo[1], ii = gi + a.halo[2];
      (void)o; (void)m; (void)ii;
      constexpr int j = 0;
%(tb_loads)s
%(tb_sub)s
%(tb_gdecl)s
      {
%(tb_coords)s
%(tb_decode)s
%(tb_collide)s
      }
%(tb_lds_stores)s
    }
    __syncthreads();
    S* tmp = cur;
    cur = nxt;
    nxt = tmp;
  }
  for (int c = threadIdx.x; c < t.tm * t.ti; c += blockDim.x) {
    const int q = divide(c, t.inv_ti);
    const int lr = t.nt * MH + q, lc = t.nt + c - q * t.ti;
    const int gm = m0 + lr, gi = i0 + lc;
    if (gm >= a.nin[1] || gi >= a.nin[2]) continue;
    const int64_t dst = (int64_t)(a.halo[0] * a.n1 + gm + a.halo[1]) * a.rs + a.lead + gi + a.halo[2];
#pragma unroll
    for (int k = 0; k < NS; ++k) fn[a.dst_off[k] + dst] = cur[k * RC + lr * RI + lc];
  }
}

"""

_PAIR_KERNEL = r"""// ------------------------------------------------ two steps per pass (3D)
// A step of a grid past the caches is bound by HBM: it reads and writes every population
// once.  This kernel advances two steps per read and write, with the per-cell arithmetic of
// fused_step (the same generated lines, so the same bits), on the wrap path.  A workgroup
// owns a column of 32 x ty cells (inner x mid axes) and walks along the outer axis.  For
// each plane its threads, one per cell of the column and a halo of one cell around it, pull
// and collide the first step into LDS; the column's own threads then do the second step
// of the plane before, whose pulls from below, in and above are all there: two planes of
// the upward populations, one of the level and one of the downward ones.  The next
// plane's pulls are in flight meanwhile.  Folded bounce-back copies read the own cell
// instead (MASK), in both steps.
// 32 cells are 128 B of FP32; 13 rows and their halo are 510 of 512 threads, two
// workgroups to a CU in 128 registers.  FP64 needs more registers (two workgroups: 75
// spilled, 605 us per step of 150 x 201 x 183) and has a CU for one workgroup of 16 rows in
// 168, with folded links 13 rows in 256.  What bounds it now: 256^3 FP32 at 308 us per step
// moves 4.4 TB/s of HBM traffic (1.1 reads and 1 write per population and two steps) with
// the vector units under half busy; the rest are the barriers of two workgroups per CU.
template <typename C>
struct PairArgs {
  int32_t tiles_i, tiles_m, ty, nz;   // tiles along the inner and mid axes, rows of a tile, planes per workgroup
  C times[2];                     // t of each step
};

constexpr int PAIR_TX = 32, PAIR_RX = PAIR_TX + 2;

template <typename S, bool MASK>
constexpr int pair_rows() {
  return sizeof(S) == 8 && !MASK ? 16 : 13;
}
template <int TY>
constexpr int pair_threads() {
  return ((TY + 2) * PAIR_RX + 63) / 64 * 64;
}
template <typename S, bool MASK, int TY>
constexpr int pair_waves() {
  return sizeof(S) == 8 ? (pair_threads<TY>() + 255) / 256 : 2 * pair_threads<TY>() / 256;
}
template <typename S, int TY>
constexpr size_t pair_lds() {
  return sizeof(S) * (2 * PAIR_UP + PAIR_LEVEL + PAIR_DOWN) * (TY + 2) * PAIR_RX;
}

__device__ __forceinline__ int pair_wrap(int x, int n) {
  x += (x < 0) ? n : 0;
  x -= (x >= n) ? n : 0;
  x -= (x >= n) ? n : 0;
  return x;
}

// a uniform value that the compiler must take as new in every pass of the loop: without
// it the address of every population's slot is kept in two registers across the loop
template <typename T>
__device__ __forceinline__ T opaque(T x) {
  asm volatile("" : "+s"(x));
  return x;
}

template <typename S>
__device__ __forceinline__ S buffer_load(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
  S x;
  if constexpr (sizeof(S) == 8) {
    const auto b = __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0);
    __builtin_memcpy(&x, &b, 8);
  } else {
    const auto b = __builtin_amdgcn_raw_buffer_load_b32(r, v, s, 0);
    __builtin_memcpy(&x, &b, 4);
  }
  return x;
}
// the value of a load, waited for here
template <typename S>
__device__ __forceinline__ S arrived(S x) {
  typename Bits<S>::T b;
  __builtin_memcpy(&b, &x, sizeof(S));
  asm volatile("" : "+v"(b));
  __builtin_memcpy(&x, &b, sizeof(S));
  return x;
}

// the collision of fused_step for one cell (the same generated lines, so the same bits)
template <typename S>
__device__ __forceinline__ void pair_collide(const S (&L)[NS], S (&G)[NS],
                                             const StepArgs<typename Codec<S>::C>& a, int o, int m, int ii,
                                             typename Codec<S>::C tt) {
  using C = typename Codec<S>::C;
  constexpr bool DEV = Codec<S>::kind != LBM_F64;
  constexpr int j = 0;
  const C half_dt = a.half_dt;
  const C* one_minus = a.one_minus;
  const C* omega = a.omega;
  const C* cref = a.cref;
  (void)half_dt; (void)tt; (void)cref; (void)j; (void)o; (void)m; (void)ii; (void)one_minus; (void)omega;
%(pair_coords)s
%(pair_decode)s
%(pair_collide)s
}

template <typename S, bool MASK, int TY>
__global__ void __launch_bounds__(pair_threads<TY>()) __attribute__((amdgpu_waves_per_eu(pair_waves<S, MASK, TY>())))
pair_step(const S* __restrict__ f, S* __restrict__ fn, const StepArgs<typename Codec<S>::C> a,
          const PairArgs<typename Codec<S>::C> t) {
  constexpr int RX = PAIR_RX, RY = TY + 2, R = RX * RY;
  extern __shared__ double pair_smem[];
  S* const up = reinterpret_cast<S*>(pair_smem);   // [2][PAIR_UP][R]
  S* const level = up + 2 * PAIR_UP * R;           // [PAIR_LEVEL][R]
  S* const down = level + PAIR_LEVEL * R;          // [PAIR_DOWN][R]
  const int total = gridDim.x, xcd = blockIdx.x %% 8;
  const int lin = xcd * (total / 8) + min(xcd, total %% 8) + (int)blockIdx.x / 8;
  const int i0 = lin %% t.tiles_i * PAIR_TX, m0 = lin / t.tiles_i %% t.tiles_m * t.ty;
  const int z0 = lin / (t.tiles_i * t.tiles_m) * t.nz, z1 = min(z0 + t.nz, a.nin[0]);
  const int c = threadIdx.x, e = c - RY * PAIR_TX;
  const int ry = min(e < 0 ? c / PAIR_TX : e >> 1, t.ty + 1);   // the threads past the last row repeat it
  const bool active = c < R;
  const int rx = e < 0 ? 1 + c %% PAIR_TX : (e & 1) * (RX - 1);
  const int at = ry * RX + rx;
  const int gm = pair_wrap(m0 - 1 + ry, a.nin[1]), gi = pair_wrap(i0 - 1 + rx, a.nin[2]);
  const bool owner = e < 0 && ry >= 1 && ry <= t.ty && m0 + ry <= a.nin[1] && i0 + rx <= a.nin[2];
  const uint64_t plane = (uint64_t)a.n1 * a.rs * sizeof(S);
  const uint32_t pop = NS > 1 ? (uint32_t)(a.dst_off[1] * sizeof(S)) : 0u;
  // byte offsets inside one plane of one population, of the cell and the cells it pulls from
%(pair_lat)s
  const uint32_t* const mask = MASK ? a.bbmask + (int64_t)gm * a.nin[2] + gi : nullptr;
  const int64_t mplane = (int64_t)a.nin[1] * a.nin[2];
  S P[NS];
  const auto fetch = [&](int p, uint32_t bits) {
    const int op = pair_wrap(p, a.nin[0]);
    const uint64_t z_0 = (op + a.halo[0]) * plane;
    const uint64_t z_p1 = (pair_wrap(op - 1, a.nin[0]) + a.halo[0]) * plane;
    const uint64_t z_n1 = (pair_wrap(op + 1, a.nin[0]) + a.halo[0]) * plane;
    const auto r_0 = buffer(f, z_0), r_p1 = buffer(f, z_p1), r_n1 = buffer(f, z_n1), r_f = buffer(f, 0);
    uint32_t kb = opaque(0u);
    (void)z_0; (void)z_p1; (void)z_n1;
    if (MASK && __ballot(bits != 0)) {
%(pair_fetch_mask)s
    } else {
%(pair_fetch)s
    }
  };
  const auto maskword = [&](int p) { return mask[pair_wrap(p, a.nin[0]) * mplane]; };
  uint32_t b_p = 0, b_c = 0, b_n = 0;   // mask words of planes p - 1, p, p + 1
  if (MASK) {
    b_c = maskword(z0 - 1);
    b_n = maskword(z0);
  }
  fetch(z0 - 1, b_c);
  for (int p = z0 - 1; p <= z1; ++p) {
    S L[NS], G[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) L[k] = P[k];
    uint32_t b_nn = 0;
    if (p < z1) {
      fetch(p + 1, b_n);
      if (MASK && p + 1 < z1) b_nn = maskword(p + 2);
    }
    pair_collide<S>(L, G, a, pair_wrap(p, a.nin[0]) + a.halo[0], gm + a.halo[1], gi + a.halo[2], t.times[0]);
    // the second step at plane p - 1: what lies below it and in it
    const bool second = p > z0 && owner;
    S* const up_p = up + (p & 1) * PAIR_UP * R;
    const S* const up_1 = up + (p & 1 ^ 1) * PAIR_UP * R;
    (void)up_1;
    if (second) {
%(pair_read1)s
    }
    __syncthreads();
    if (active) {
%(pair_write)s
    }
    __syncthreads();
    if (second) {
%(pair_read2)s
      pair_collide<S>(L, G, a, p - 1 + a.halo[0], gm + a.halo[1], gi + a.halo[2], t.times[1]);
    }
    // the next plane is waited for before the stores: behind them the wait would be for
    // the stores as well
#pragma unroll
    for (int k = 0; k < NS; ++k) P[k] = arrived(P[k]);
    if (second) {
      const auto r_out = buffer(fn, (p - 1 + a.halo[0]) * plane);
      const auto store = [&](auto nt) {
        constexpr bool NT = decltype(nt)::value;
        uint32_t kb = opaque(0u);
%(pair_store)s
      };
      if (a.nt) store(std::true_type{});
      else store(std::false_type{});
    }
    if (MASK) {
      b_p = b_c;
      b_c = b_n;
      b_n = b_nn;
    }
  }
  (void)b_p;
}

"""

_PAIR_LAUNCH = r"""template <typename S, bool MASK>
static int pair_launch(const void* f, void* fn, const lbm_layout* L, lbm_params* p, int nz, hipStream_t s) {
  using C = typename Codec<S>::C;
  constexpr int TY = pair_rows<S, MASK>();
  StepArgs<C> a;
  int rc = make_args<C>(L, p, &a);
  if (rc) return rc;
  PairArgs<C> t{};
  t.tiles_i = (a.nin[2] + PAIR_TX - 1) / PAIR_TX;
  t.tiles_m = (a.nin[1] + TY - 1) / TY;
  t.ty = (a.nin[1] + t.tiles_m - 1) / t.tiles_m;
  t.nz = nz;
  a.nt = stream_stores(L, 256);
  for (int q = 0; q < 2; ++q) {
    t.times[q] = (C)p->t;
    p->t += p->dt;
  }
  const size_t lds = pair_lds<S, TY>();
  const unsigned groups = (unsigned)(t.tiles_i * t.tiles_m * ((a.nin[0] + nz - 1) / nz));
  const auto kernel = pair_step<S, MASK, TY>;
  if (lds > 64 * 1024)
    LBM_CHECK_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  kernel<<<groups, pair_threads<TY>(), lds, s>>>((const S*)f, (S*)fn, a, t);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

// Planes per workgroup of the two-step kernel on this grid, or 0: one step at a time.
// The choice is between whole runs of one step per launch at 5.6 TB/s of reads and writes
// plus 2 us, and the least estimate of the two-step kernel over the numbers of chunks
// along the outer axis: nz + 2 planes per workgroup at so many us per plane with few
// workgroups, one or two on every CU, a little more in long chunks, whose neighbours
// drift apart in the L2 (constants fitted to a sweep of 19 grids, 80^3 to 256^3, with and
// without folded links, FP32 and FP64 D3Q19 on MI355X: 5 %% rms).  Per step, one at a time /
// two: 256^3 FP32 448 / 308 us, 128^3 53 / 48, 80^3 16 / 19; 150 x 201 x 183 FP64 310 / 206,
// 96^3 45 / 35; 256 x 128 x 128 with spheres FP32 118 / 100, FP64 222 / 174; 200^3 D3Q15 FP32
// 192 / 142, FP64 335 / 238, D3Q6 FP32 70 / 56, FP64 131 / 89.
template <typename S, bool MASK>
static int pair_planes(const int32_t (&nin)[3]) {
  constexpr double part = NS / 19.0;
  constexpr double few = part * (sizeof(S) == 8 ? (MASK ? 4.3 : 4.9) : 2.9);
  constexpr double one = part * (sizeof(S) == 8 ? (MASK ? 6.6 : 7.7) : 4.1), two = part * 7.0;
  constexpr double drift = MASK ? 0.006 : 0.0008, start = MASK ? 5.0 : 1.0;
  const int64_t tiles = (int64_t)((nin[2] + PAIR_TX - 1) / PAIR_TX) *
                        ((nin[1] + pair_rows<S, MASK>() - 1) / pair_rows<S, MASK>());
  double best = 0.9 * 2.0 * (2.0 + (double)nin[0] * nin[1] * nin[2] * NS * 2.0 * sizeof(S) / 5.6e6);
  int planes = 0;
  for (int chunks = 1; chunks <= nin[0] / 4; ++chunks) {
    const int nz = (nin[0] + chunks - 1) / chunks;
    const int64_t groups = tiles * ((nin[0] + nz - 1) / nz), cap = sizeof(S) == 8 ? 256 : 512;
    const int64_t rest = groups %% cap;
    double us = (double)(groups / cap) * (sizeof(S) == 8 ? one : two);
    if (rest > 256) us += two * (0.85 + 0.15 * (double)(rest - 256) / 256.0);
    else if (rest > 0) us += few + (one - few) * (double)rest / 256.0;
    us = start + (nz + 2) * (1.0 + drift * nz) * us;
    if (us < best) {
      best = us;
      planes = nz;
    }
  }
  return planes;
}

// whether the compiler spilled more than a few registers of the kernel to scratch memory: a
// reload there waits for every load in flight (200^3 D3Q19 FP64, us per step one at a time /
// in pairs: source terms in t, 12 B spilled, 420 / 315; linear in X, Y and Z, 8 B, 421 / 354; sines
// of X, Y, Z and t, 44 B, 421 / 468)
template <typename S, bool MASK>
static bool pair_spills() {
  static const bool spills = [] {
    hipFuncAttributes at;
    const hipError_t e = hipFuncGetAttributes(&at, (const void*)pair_step<S, MASK, pair_rows<S, MASK>()>);
    if (e != hipSuccess) (void)hipGetLastError();   // single steps; not the next launch's error
    return e != hipSuccess || at.localSizeBytes > 24;
  }();
  return spills;
}

// one launch of the two-step kernel, where it is the faster one (*done)
template <typename S, bool MASK>
static int pair_try(const void* f, void* fn, const lbm_layout* L, lbm_params* p, bool* done, hipStream_t s) {
  // an offset inside a plane (with folded links inside the array) has 32 bits
  const int64_t reach = ((NS - 1) * L->pop_stride + (MASK ? L->n[0] : 1) * L->n[1] * L->row_stride) * (int64_t)sizeof(S);
  int32_t nin[3];
  for (int d = 0; d < 3; ++d) nin[d] = (int32_t)(L->n[d] - 2 * L->halo[d]);
  if (pair_lds<S, pair_rows<S, MASK>()>() > 160 * 1024 || reach >= ((int64_t)1 << 32) - (1 << 20) || nin[0] < 4 || nin[1] < 32 || nin[2] < 32) return 0;
  const int nz = pair_planes<S, MASK>(nin);
  if (nz == 0 || pair_spills<S, MASK>()) return 0;
  *done = true;
  return pair_launch<S, MASK>(f, fn, L, p, nz, s);
}

static int pair_any(const void* f, void* fn, const lbm_layout* L, lbm_params* p, bool* done, hipStream_t s) {
  *done = false;
  // folded links beyond copies (a table), a launch shape asked for, or 2-byte formats (bound
  // by arithmetic: 128^3 FP16 33 us per step one at a time, 40 us in pairs): single steps
  if (p->bbtab_bits || p->vec_cells != 0 || p->xcd_remap >= 0 || p->single_steps) return 0;
  switch (L->storage) {
    case LBM_F64: return p->bbmask ? pair_try<double, true>(f, fn, L, p, done, s) : pair_try<double, false>(f, fn, L, p, done, s);
    case LBM_F32: return p->bbmask ? pair_try<float, true>(f, fn, L, p, done, s) : pair_try<float, false>(f, fn, L, p, done, s);
    case LBM_F32D: return p->bbmask ? pair_try<f32dev, true>(f, fn, L, p, done, s) : pair_try<f32dev, false>(f, fn, L, p, done, s);
  }
  return 0;
}

"""

_TB_LAUNCH = r"""// one launch of tb_step: nt steps of every tile; advances params->t by nt dt
template <typename S>
static int tb_launch(void* f, void* fn, const lbm_layout* L, lbm_params* p, int nt, int tm, int ti,
                     hipStream_t s) {
  using C = typename Codec<S>::C;
  StepArgs<C> a;
  int rc = make_args<C>(L, p, &a);
  if (rc) return rc;
  LBM_REQUIRE(a.nin[1] >= tm && a.nin[2] >= ti && (DIM == 1 || a.nin[1] >= nt) && a.nin[2] >= nt,
              "tile %%d x %%d / %%d steps larger than the interior", tm, ti, nt);
  TbArgs<C> t{};
  t.nt = nt;
  t.tm = tm;
  t.ti = ti;
  t.tiles_i = (a.nin[2] + ti - 1) / ti;
  t.inv_ti = reciprocal(ti);
  for (int q = 0; q <= nt; ++q) t.inv[q] = reciprocal(ti + 2 * (nt - q));
  for (int q = 0; q < nt; ++q) {
    t.times[q] = (C)p->t;
    p->t += p->dt;
  }
  const int tiles_m = (a.nin[1] + tm - 1) / tm;
  const size_t region = (size_t)(DIM == 1 ? tm : tm + 2 * nt) * (ti + 2 * nt);
  const bool mask = TB_MASK && p->bbmask, table = mask && p->bbtab_bits;
  constexpr size_t full_plane = tb_plane<S, false>(), half_plane = tb_plane<S, true>();
  LBM_REQUIRE(region <= full_plane, "tile region of %%zu cells exceeds the %%zu cells of a plane", region, full_plane);
  const bool half = region <= half_plane;
  const size_t plane = half ? half_plane : full_plane;
  const size_t lds = 2 * NS * sizeof(S) * plane + region * ((mask ? 4 : 0) + (table ? 8 : 0));
  LBM_REQUIRE(lds <= 160 * 1024, "tile needs %%zu bytes of LDS", lds);
  // a thread per region cell, at most TB_THREADS, or half as many where two
  // workgroups share a CU
  const unsigned tiles = (unsigned)(tiles_m * t.tiles_i);
  const unsigned most = half && tiles > 256 ? TB_THREADS / 2 : TB_THREADS;
  const unsigned threads = (unsigned)(region < most ? (region + 63) / 64 * 64 : most);
  const void* kernel = half ? (const void*)tb_step<S, true> : (const void*)tb_step<S, false>;
  LBM_CHECK_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  if (half) tb_step<S, true><<<dim3(tiles), dim3(threads), lds, s>>>((const S*)f, (S*)fn, a, t);
  else tb_step<S, false><<<dim3(tiles), dim3(threads), lds, s>>>((const S*)f, (S*)fn, a, t);
  LBM_CHECK_HIP(hipGetLastError());
  return 0;
}

#define LBM_DISPATCH_BLOCKED(kind, FN, f, fn, L, p, nt, tm, ti, s, rc)          \
  do {                                                                          \
    switch (kind) {                                                             \
      case LBM_F64: rc = FN<double>(f, fn, L, p, nt, tm, ti, s); break;         \
      case LBM_F32: rc = FN<float>(f, fn, L, p, nt, tm, ti, s); break;          \
      case LBM_F16D: rc = FN<_Float16>(f, fn, L, p, nt, tm, ti, s); break;      \
      case LBM_BF16D: rc = FN<::lbm::bf16>(f, fn, L, p, nt, tm, ti, s); break;  \
      case LBM_F32D: rc = FN<::lbm::f32dev>(f, fn, L, p, nt, tm, ti, s); break; \
      default: ::lbm::set_error("unknown storage kind %%d", (int)(kind)); rc = -1; \
    }                                                                           \
  } while (0)

"""

# 3D / 1D schemes: no temporally blocked kernel
_TB_LAUNCH_NONE = r"""#define LBM_DISPATCH_BLOCKED(kind, FN, f, fn, L, p, nt, tm, ti, s, rc) \
  do {                                                                \
    (void)(kind);                                                     \
    rc = 0;                                                           \
  } while (0)

"""


def _pair_source(vel, ksym, decode, coords, collide):
    """The kernel that advances a 3D scheme with velocity components in {-1, 0, 1} by two
    steps per pass over memory."""
    ns = len(vel)
    arr = lambda lines: [re.sub(r"\b([LG])(\d+)\[j\]", r"\1[\2]", ln) for ln in lines]   # noqa: E731
    nm = lambda c: ("p%d" % c) if c > 0 else ("n%d" % -c if c < 0 else "0")   # noqa: E731
    slot = {}
    for name, v0 in (("up", 1), ("level", 0), ("down", -1)):
        ks = [k for k in range(ns) if vel[k][0] == v0]
        slot.update({k: (name, q) for q, k in enumerate(ks)})
    count = {n: max([q + 1 for m, q in slot.values() if m == n], default=0) for n in ("up", "level", "down")}
    lat = []
    for d, axis, n, step in ((1, "gm", 1, "(uint32_t)a.rs"), (2, "gi", 2, "1u")):
        for c in sorted({v[d] for v in vel} | {0}):
            extra = " + (uint32_t)(a.lead + a.halo[2])" if d == 2 else ""
            halo = " + a.halo[1]" if d == 1 else ""
            lat.append("  const uint32_t s%d_%s = ((uint32_t)(pair_wrap(%s - (%d), a.nin[%d])%s) * %s%s) * (uint32_t)sizeof(S);"
                       % (d, nm(c), axis, c, n, halo, step, extra))
    offs = sorted({v[1:] for v in vel} | {(0, 0)})
    lat += ["  const uint32_t o_%s_%s = s1_%s + s2_%s;" % (nm(a), nm(b), nm(a), nm(b)) for a, b in offs]
    ref = lambda k: "o_%s_%s" % (nm(vel[k][1]), nm(vel[k][2]))   # noqa: E731
    # kb runs over the populations (opaque: the compiler would multiply again for each)
    fetch, fetch_mask = [], []
    for k in range(ns):
        step = "" if k == 0 else "      kb = opaque(kb + pop);\n"
        load = "      P[%d] = buffer_load<S>(r_%s, %s, kb);" % (k, nm(vel[k][0]), ref(k))
        fetch.append(step + load)
        if ksym is not None and ksym[k] != k:
            fetch_mask.append(step + "      P[%d] = buffer_load<S>(r_f, (bits & %du) ? o_0_0 + (%du * pop + (uint32_t)z_0) :"
                              " %s + (kb + (uint32_t)z_%s), 0u); __builtin_amdgcn_sched_barrier(0);"
                              % (k, 1 << k, ksym[k], ref(k), nm(vel[k][0])))
        else:
            fetch_mask.append(step + load)
    read1, write, read2, store = [], [], [], []
    for k in range(ns):
        name, q = slot[k]
        near = "[%d * R + at - (%d)]" % (q, vel[k][1] * 34 + vel[k][2])
        write.append("      %s[%d * R + at] = G[%d];" % ("up_p" if name == "up" else name, q, k))
        bounce = ksym is not None and ksym[k] != k
        if bounce:
            # population ksym at the own cell after the first step: planes p - 1 of LDS,
            # before plane p is written
            oname, oq = slot[ksym[k]]
            own = "%s[%d * R + at]" % ("up_1" if oname == "up" else oname, oq)
        if name == "down":
            if bounce:
                read1.append("      if (MASK && (b_p & %du)) L[%d] = %s;" % (1 << k, k, own))
            read2.append("      %sL[%d] = down%s;" % ("if (!MASK || !(b_p & %du)) " % (1 << k) if bounce else "", k, near))
        else:
            x = ("up_p" if name == "up" else name) + near
            read1.append("      L[%d] = %s%s;" % (k, "(MASK && (b_p & %du)) ? %s : " % (1 << k, own) if bounce else "", x))
    for k in range(ns):
        store.append("        buffer_store<S, NT>(r_out, o_0_0, kb, G[%d]);" % k
                     + (" kb = opaque(kb + pop);" if k < ns - 1 else ""))
    j = "\n".join
    return (_PAIR_KERNEL % dict(
        pair_coords=_indent(coords), pair_decode=_indent(arr(decode)), pair_collide=_indent(arr(collide)),
        pair_lat=j(lat), pair_fetch_mask=j(fetch_mask), pair_fetch=j(fetch), pair_read1=j(read1),
        pair_write=j(write), pair_read2=j(read2), pair_store=j(store))
        ).replace("PAIR_UP", str(count["up"])).replace("PAIR_LEVEL", str(count["level"])).replace(
            "PAIR_DOWN", str(count["down"]))


def _indent(lines, n=2):
    return "\n".join(" " * n + ln for ln in lines)


def generate_source(spec: KernelSpec) -> str:
    ns, dim = spec.ns, spec.dim
    vel = [_canon(v, dim) for v in spec.velocities]
    ksym = _pairs(spec)
    sig_f2m = _row_parities(spec.M, ksym, by_rows=True) if ksym else None
    sig_m2f = None
    if ksym and sig_f2m:
        sig_cols = _row_parities(spec.invM, ksym, by_rows=False)
        sig_m2f = sig_cols if sig_cols == sig_f2m else None
        if sig_m2f is None:
            sig_f2m = None
    M = [[Fraction(c) for c in r] for r in spec.M]
    iM = [[Fraction(c) for c in r] for r in spec.invM]
    fvars = ["f%d" % k for k in range(ns)]
    mvars = ["m%d" % i for i in range(ns)]

    # ---------------------------------------------------------- fused step
    # folded link lists: where bit k of the cell's mask word is set, the pulled
    # value of population k is what the link f[k, x - v_k] = sign f[ksym, x] + value
    # would have stored, computed as links_kernel computes it: a copy of f[ksym, x]
    # for sign 1 without a value, else decode_dev of the table entry's source,
    # r = sign v, r += value, encode (w = 0); bit 31 of the mask word marks the
    # cells that have table entries (ns <= 31).
    # The entries go in batches of directions whose loads do not depend on each other's
    # values (a lane without the entry reads its cell's first).  Direction after
    # direction, each waiting for entry and source, a lid cell's three links made every
    # step of a 64^2 FP64 cavity wait (5.5 us; 4.7 this way).
    bbsub = []
    if ksym is not None:
        bbsub = ["{",
                 "  if (a.bbmask) {",
                 "    using CC = typename Codec<S>::C;",
                 "    const int64_t mc = ((int64_t)oo * a.nin[1] + mm) * a.nin[2] + i;",
                 "#pragma unroll",
                 "    for (int j = 0; j < VEC; ++j) {",
                 "      const uint32_t bits = a.bbmask[mc + j];",
                 "      if (bits) {"]
        for k in range(ns):
            if ksym[k] != k:
                bbsub.append("        if (bits & %du) L%d[j] = f[(I)a.dst_off[%d] + cell + j];" % (1 << k, k, ksym[k]))
        bbsub += ["        if constexpr (TABLE) {",
                  "        uint32_t tb = 0, tbase = 0;",
                  "        if (bits & 0x80000000u) {",
                  "          tb = a.bbtab_bits[mc + j];",
                  "          tbase = a.bbtab_base[mc + j];",
                  "        }",
                  "        (void)tbase;"]
        # directions that leave through the same face together: its cells need one or two
        linked = sorted((k for k in range(ns) if ksym[k] != k), key=lambda k: vel[k])
        size = 8 if ns <= 9 else 3
        for batch in (linked[q:q + size] for q in range(0, len(linked), size)):
            every = sum(1 << k for k in batch)
            bbsub.append("        if (tb & %du) {" % every)
            for k in batch:
                bit = 1 << k
                bbsub.append("          const uint32_t e%d = (tb & %du) ? tbase + (uint32_t)__builtin_popcount(tb & %du) : tbase;"
                             % (k, bit, bit - 1))
            for k in batch:
                bbsub += ["          const uint32_t s%d = a.bbtab_src[e%d];" % (k, k),
                          "          const CC a%d = a.bbtab_sign[e%d], r%d = a.bbtab_rhs[e%d];" % (k, k, k, k)]
            bbsub += ["          const S v%d = f[s%d];" % (k, k) for k in batch]
            bbsub.append("          if (a.bbtab_src2) {")
            for k in batch:
                bbsub += ["            const uint32_t t%d = a.bbtab_src2[e%d];" % (k, k),
                          "            const CC c%d = a.bbtab_c2[e%d];" % (k, k)]
            bbsub += ["            const S w%d = f[t%d == 0xffffffffu ? s%d : t%d];" % (k, k, k, k) for k in batch]
            for k in batch:
                bbsub += ["            if (tb & %du) {" % (1 << k),
                          "              CC r_ = a%d * Codec<S>::decode_dev(v%d, (CC)0);" % (k, k),
                          "              r_ = t%d == 0xffffffffu ? r_ : r_ + c%d * Codec<S>::decode_dev(w%d, (CC)0);" % (k, k, k),
                          "              r_ += r%d;" % k,
                          "              L%d[j] = Codec<S>::encode(r_, (CC)0);" % k,
                          "            }"]
            bbsub.append("          } else {")
            for k in batch:
                bbsub += ["            if (tb & %du) {" % (1 << k),
                          "              CC r_ = a%d * Codec<S>::decode_dev(v%d, (CC)0);" % (k, k),
                          "              r_ += r%d;" % k,
                          "              L%d[j] = Codec<S>::encode(r_, (CC)0);" % k,
                          "            }"]
            bbsub += ["          }", "        }"]
        bbsub += ["        }", "      }", "    }", "  }", "}"]
    loads = ["S %s;" % ", ".join("L%d[VEC]" % k for k in range(ns))]
    loads.append("if (!FOLD) {")
    for k in range(ns):
        loads.append("  vload_pull<S, VEC, %d>(L%d, f + ((I)a.src_off[%d] + (%d) + cell));" % (-vel[k][2], k, k, vel[k][2]))
    loads.append("} else {")
    # wrapped outer / mid coordinates per distinct component value; the contiguous
    # axis is wrapped per element, only for the vectors that straddle the row ends
    comps = [sorted({v[d] for v in vel}) for d in range(2)]
    names = {}
    for d, axis in enumerate(("o", "m")):
        for c in comps[d]:
            nm = "w%d_%s" % (d, ("p%d" % c) if c >= 0 else ("n%d" % -c))
            names[(d, c)] = nm
            loads.append("  int %s = %s - (%d);" % (nm, axis, c))
            loads.append("  %s += (%s < a.halo[%d]) ? a.nin[%d] : 0;" % (nm, nm, d, d))
            loads.append("  %s -= (%s >= a.halo[%d] + a.nin[%d]) ? a.nin[%d] : 0;" % (nm, nm, d, d, d))
    for k, (v0, v1, v2) in enumerate(vel):
        loads.append("  {")
        loads.append("    const I row = (I)a.dst_off[%d] + ((I)%s * a.n1 + %s) * a.rs + a.lead;"
                     % (k, names[(0, v0)], names[(1, v1)]))
        loads.append("    const int s0 = ii - (%d);" % v2)
        if v2 == 0:
            loads.append("    vload<S, VEC>(L%d, f + (row + s0));" % k)
        else:
            loads.append("    if (s0 >= a.halo[2] && s0 + VEC <= a.halo[2] + a.nin[2]) {")
            loads.append("      vload_pull<S, VEC, %d>(L%d, f + (row + ii));" % (-v2, k))
            loads.append("    } else {")
            loads.append("      for (int j = 0; j < VEC; ++j) {")
            loads.append("        int c = s0 + j;")
            loads.append("        c += (c < a.halo[2]) ? a.nin[2] : 0;")
            loads.append("        c -= (c >= a.halo[2] + a.nin[2]) ? a.nin[2] : 0;")
            loads.append("        L%d[j] = f[row + c];" % k)
            loads.append("      }")
            loads.append("    }")
        loads.append("  }")
    loads.append("}")
    gdecl = ["S %s;" % ", ".join("G%d[VEC]" % k for k in range(ns))]
    rel = spec.rel_vel is not None
    if rel:
        # relative-velocity schemes collide full values in every format
        decode = ["C f%d = Codec<S>::decode(L%d[j], a.wshift[%d]);" % (k, k, k) for k in range(ns)]
    else:
        decode = ["C f%d = DEV ? Codec<S>::decode_dev(L%d[j], a.wshift[%d]) : Codec<S>::decode(L%d[j], a.wshift[%d]);"
                  % (k, k, k, k, k) for k in range(ns)]
    vstores = ["vstore<S, VEC, NT>(fn + ((I)a.dst_off[%d] + cell), G%d);" % (k, k) for k in range(ns)]

    # The arithmetic of the step.  Contracted, moments share partial sums and a product and a
    # sum of one statement become one FMA: up to a quarter fewer instructions.  Errors
    # against wider arithmetic, replayed on the CPU over 32 to 128 flows of 30 to 400 steps,
    # relative to single roundings (density, momentum):
    #   FP64 0.74, 0.83 (D3Q19), 0.97, 0.96 (D2Q9): contracted; 128^3 in pairs 84 -> 78 us;
    #   FP32 in 3D 0.99, 0.99: contracted, and the increment is added to the stored value
    #   itself; 256^3 in pairs 308 -> 305 us per step, 80^3 15.7 -> 15.2;
    #   2-byte formats in 3D 1.01, 1.00: contracted but for M^-1 m, where a product enters several
    #   populations and, fused, rounds differently in each of their sums; 128^3 27.0 -> 25.2 us;
    #   FP32 deviations in 3D 1.05, 1.07 (shared sums alone 1.07, 1.03; 256^3 Taylor-Green vortex
    #   after 1000 steps 4.7e-7 against 3.9e-7): not contracted, their accuracy is that of
    #   their arithmetic, and it costs them nothing (306 us per step of 256^3 either way).
    # The FP32-compute formats of 1D and 2D schemes are not contracted either and keep the
    # results they have always had bit for bit (contracted: momentum 0.97 FP32, 0.99
    # deviations; 1024 x 256 channel 634 us per 200 steps instead of 670).
    fuse, fuse_dev = not rel, not rel and dim == 3

    def step_lines(dev, on, on_back, added=False):
        """f2m, collision and m2f of one cell in deviations (dev) or full values, f2m and
        collision contracted (on), m2f contracted (on_back); added: the increments are
        added to the stored values."""
        b1 = _SumBuilder("p", on)
        f2m = _transform(b1, M, fvars, mvars, ksym, sig_f2m)
        out = (["#pragma clang fp contract(on)"] if on else []) + b1.lines + ["C %s = %s;" % (o, e) for o, e in f2m]
        if rel:
            coll, names = _relative_collision_lines(spec)
        elif dev:
            coll, names = _deviation_collision_lines(spec, on)
        else:
            coll, names = _collision_lines(spec, with_sources=True, fuse=on), mvars
        dev = dev and not rel
        b2 = _SumBuilder("rd" if dev else "r", on)
        m2f = _inverse_transform(b2, iM, names, ["g%d" % k for k in range(ns)], ksym, sig_m2f, tag="d" if dev else "")
        back = b2.lines + ["const C %s = %s;" % (o, e) for o, e in m2f]
        form = "L{0}[j] + g{0}" if added else \
            "Codec<S>::encode_dev(f{0} + g{0}, a.wshift[{0}])" if dev else "Codec<S>::encode(g{0}, a.wshift[{0}])"
        back += [("G{0}[j] = " + form + ";").format(k) for k in range(ns)]
        return out + coll + (["{", "#pragma clang fp contract(off)"] + back + ["}"] if on and not on_back else back)

    cases = [("DEV", step_lines(True, False, False)), (None, step_lines(False, fuse, fuse))]
    if fuse_dev:
        cases = [("Codec<S>::kind == LBM_F32D", step_lines(True, False, False)),
                 ("Codec<S>::kind == LBM_F32", step_lines(True, True, True, added=True)),
                 ("DEV", step_lines(True, True, False)), cases[1]]
    collide = []
    for test, lines in cases:
        collide.append(("} else " if collide else "") + ("if constexpr (%s) {" % test if test else "{"))
        collide += ["  " + ln for ln in lines]
    collide.append("}")

    # ---------------------------------------------------------- f2m / m2f / eq
    b3 = _SumBuilder("p")
    f2m_full_lines = _transform(b3, M, fvars, mvars, ksym, sig_f2m)
    f2m_loads = ["const C f%d = Codec<S>::widen(f[%d * fl.pop_stride + cf], (double)a.wshift[%d]);" % (k, k, k)
                 for k in range(ns)]
    f2m_full = b3.lines + ["const C %s = %s;" % (o, e) for o, e in f2m_full_lines]
    f2m_stores = ["mo[%d * ml.pop_stride + cm] = m%d;" % (i, i) for i in range(ns)]

    b4 = _SumBuilder("r")
    m2f_full_lines = _inverse_transform(b4, iM, mvars, ["g%d" % k for k in range(ns)], ksym, sig_m2f)
    m2f_loads = ["const C m%d = mi[%d * ml.pop_stride + cm];" % (i, i) for i in range(ns)]
    m2f_full = b4.lines + ["const C %s = %s;" % (o, e) for o, e in m2f_full_lines]
    m2f_stores = ["Codec<S>::store(f, %d * fl.pop_stride + cf, (typename Codec<S>::C)g%d, (typename Codec<S>::C)a.wshift[%d]);" % (k, k, k)
                  for k in range(ns)]

    eq_loads = ["C m%d = mo[%d * ml.pop_stride + cm];" % (i, i) for i in range(ns)]
    eq_body = _equilibrium_lines(spec)
    eq_stores = ["mo[%d * ml.pop_stride + cm] = m%d;" % (i, i) for i in range(spec.nconsm, ns)]
    eq_loads += ["(void)m%d;" % i for i in range(spec.nconsm, ns)]
    # the fused kernel loads only the conserved rows; the equilibrium assigns the others
    eqm2f_loads = (["C m%d = mo[%d * ml.pop_stride + cm];" % (i, i) for i in range(spec.nconsm)]
                   + ["C m%d;" % i for i in range(spec.nconsm, ns)])
    eqm2f_opaque = ["m%d = stored_moment(m%d);" % (i, i) for i in range(spec.nconsm, ns)]

    # split routines: relaxation (every relaxed row) and source_term (the source rows)
    relaxed_rows = [i for i in range(spec.nconsm, ns) if spec.s[i] != 0]
    rx_loads = ["C m%d = mo[%d * ml.pop_stride + cm];" % (i, i) for i in range(ns)]
    rx_loads += ["(void)m%d;" % i for i in range(ns)]
    rx_body = _collision_lines(spec, with_sources=False)
    rx_stores = ["mo[%d * ml.pop_stride + cm] = m%d;" % (i, i) for i in relaxed_rows]
    st_loads = list(rx_loads)
    st_body = ["m%d = m%d + half_dt * (%s);" % (idx, idx, _ccode(sp.sympify(expr))) for idx, expr in spec.sources]
    st_stores = ["mo[%d * ml.pop_stride + cm] = m%d;" % (idx, idx) for idx in sorted({i for i, _ in spec.sources})]

    # cell-centre coordinates of the reference axes the source terms use (pylbm's X, Y, Z)
    used = set()
    for _, e in spec.sources:
        used |= {str(x) for x in sp.sympify(e).free_symbols}
    canon_index = ["o", "m", "(ii + j)"]
    coords = ["const C xc%d = a.xorg[%d] + a.dx * (C)%s;" % (d, d, canon_index[3 - dim + d])
              for d in range(dim) if "XYZ"[d] in used]
    vel_txt = ", ".join("{%d, %d, %d}" % v for v in vel)

    # ------------------------------------------- temporally blocked kernel (2D)
    if dim <= 2:
        tb_loads = ["S %s;" % ", ".join("L%d[1]" % k for k in range(ns))]
        tb_loads += ["L%d[0] = cur[%d * RC + lcell - (%d * RI + %d)];" % (k, k, vel[k][1], vel[k][2])
                     for k in range(ns)]
        tb_sub, tb_mask, tb_collect, tb_entries, tb_apply = [], [], [], [], []
        if ksym is not None:
            # the links of every cell that the region updates (all but its outermost
            # cells), listed as {slot | cell << 16, source} or, for a table entry,
            # {slot | cell << 16, 1 << 31 | entry}
            inner = "c - lr * RI > 0 && c - lr * RI < RI - 1" + (" && lr > 0 && lr < RW - 1" if dim == 2 else "")
            tb_mask = ["if (masked && %s) bits_[b] = a.bbmask[(int64_t)gm * a.nin[2] + gi];" % inner]
            tb_collect = ["{",
                          "  const uint32_t bits = bits_[b];",
                          "  if (bits) {",
                          "    const int lr = divide(c, t.inv[0]);",
                          "    const int64_t mc = (int64_t)wrap_near(m0 + lr, a.nin[1]) * a.nin[2] + wrap_near(i0 + c - lr * RI, a.nin[2]);",
                          "    const uint32_t tb = (bits & 0x80000000u) ? a.bbtab_bits[mc] : 0u;",
                          "    const uint32_t tbase = tb ? a.bbtab_base[mc] : 0u;",
                          "    int p_ = atomicAdd(nlinks, __builtin_popcount(bits & %du));"
                          % sum(1 << k for k in range(ns) if ksym[k] != k)]
            for k in range(ns):
                if ksym[k] != k:
                    bit = 1 << k
                    tb_collect += ["    if (bits & %du) {" % bit,
                                   "      if (p_ < cap)",
                                   "        links[p_] = make_uint2((uint32_t)(%d * RC + c - (%d * RI + %d)) | ((uint32_t)c << 16),"
                                   % (k, vel[k][1], vel[k][2]),
                                   "                               (tb & %du) ? 0x80000000u | (tbase + (uint32_t)__builtin_popcount(tb & %du))"
                                   % (bit, bit - 1),
                                   "                                          : (uint32_t)(%d * RC + c));" % ksym[k],
                                   "      ++p_;",
                                   "    }"]
            tb_collect += ["  }", "}"]
            # this thread's links in registers: slot and source (16 bits each), second
            # source, kind (0: none, 1: a copy, 2: one source, 3: two), coefficients, value
            tb_entries = ["const int nlist = masked ? *nlinks : 0;",
                          "const bool dense = nlist > cap;",
                          "uint32_t l_at[TB_LINKS], l_two[TB_LINKS];",
                          "C l_a[TB_LINKS], l_b[TB_LINKS], l_r[TB_LINKS];",
                          "#pragma unroll",
                          "for (int q = 0; q < TB_LINKS; ++q) {",
                          "  const int e = q * (int)blockDim.x + (int)threadIdx.x;",
                          "  l_at[q] = l_two[q] = 0;",
                          "  l_a[q] = l_b[q] = l_r[q] = (C)0;",
                          "  if (e < nlist && !dense) {",
                          "    const uint2 w = links[e];",
                          "    if (w.y & 0x80000000u) {",
                          "      const uint32_t x = w.y & 0x7fffffffu;",
                          "      const uint32_t rel = a.bbtab_rel[x];",
                          "      const uint32_t rel2 = a.bbtab_rel2 ? a.bbtab_rel2[x] : 0u;",
                          "      l_a[q] = a.bbtab_sign[x];",
                          "      l_r[q] = a.bbtab_rhs[x];",
                          "      l_b[q] = a.bbtab_rel2 ? a.bbtab_c2[x] : (C)0;",
                          "      const int c = (int)(w.x >> 16);",
                          "      const int src = (int)(rel & 0xffu) * RC + c + ((int)((rel >> 8) & 0xffu) - 128) * RI +",
                          "                      (int)((rel >> 16) & 0xffu) - 128;",
                          "      const int src2 = (int)(rel2 & 0xffu) * RC + c + ((int)((rel2 >> 8) & 0xffu) - 128) * RI +",
                          "                       (int)((rel2 >> 16) & 0xffu) - 128;",
                          "      const bool two = (rel2 & 0x80000000u) != 0;",
                          "      l_at[q] = (w.x & 0xffffu) | ((uint32_t)src << 16);",
                          "      l_two[q] = two ? 3u | ((uint32_t)src2 << 16) : 2u;",
                          "    } else {",
                          "      l_at[q] = (w.x & 0xffffu) | (w.y << 16);",
                          "      l_two[q] = 1u;",
                          "    }",
                          "  }",
                          "}",
                          "__syncthreads();   // the list is read: nxt is free",
                          "if (dense) {",
                          "  for (int c = threadIdx.x; c < RN; c += blockDim.x) {",
                          "    const int lr = divide(c, t.inv[0]);",
                          "    const int gm = wrap_near(m0 + lr, a.nin[1]), gi = wrap_near(i0 + c - lr * RI, a.nin[2]);",
                          "    const int64_t mc = (int64_t)gm * a.nin[2] + gi;",
                          "    msk[c] = a.bbmask[mc];",
                          "    if (table) {",
                          "      tbits[c] = a.bbtab_bits[mc];",
                          "      tbase_l[c] = a.bbtab_base[mc];",
                          "    }",
                          "  }",
                          "  __syncthreads();",
                          "}"]
            # the arithmetic of fused_step's table entries (products and sums round apart)
            tb_apply = ["if (nlist && !dense) {",
                        "  S l_v[TB_LINKS];",
                        "#pragma unroll",
                        "  for (int q = 0; q < TB_LINKS; ++q) {",
                        "    if (q * (int)blockDim.x >= nlist) break;   // the same for the whole workgroup",
                        "    if (l_two[q]) {",
                        "      const S v = cur[l_at[q] >> 16];",
                        "      l_v[q] = v;",
                        "      if (l_two[q] != 1u) {",
                        "        C r_ = l_a[q] * Codec<S>::decode_dev(v, (C)0);",
                        "        if ((l_two[q] & 0xffffu) == 3u)",
                        "          r_ = r_ + l_b[q] * Codec<S>::decode_dev(cur[l_two[q] >> 16], (C)0);",
                        "        r_ += l_r[q];",
                        "        l_v[q] = Codec<S>::encode(r_, (C)0);",
                        "      }",
                        "    }",
                        "  }",
                        "  __syncthreads();",
                        "#pragma unroll",
                        "  for (int q = 0; q < TB_LINKS; ++q) {",
                        "    if (q * (int)blockDim.x >= nlist) break;",
                        "    if (l_two[q]) cur[l_at[q] & 0xffffu] = l_v[q];",
                        "  }",
                        "  __syncthreads();",
                        "}"]
            # dense regions: bounce-back copies as selects of unconditional LDS reads (one branch per
            # cell instead of one per direction), then the table links: bits and
            # first entry from LDS, the entries from memory
            tb_sub = ["if (dense) {",
                      "  const uint32_t bits = msk[lcell];",
                      "  if (bits) {"]
            for k in range(ns):
                if ksym[k] != k:
                    tb_sub += ["    {",
                               "      const S b_ = cur[%d * RC + lcell];" % ksym[k],
                               "      L%d[0] = (bits & %du) ? b_ : L%d[0];" % (k, 1 << k, k),
                               "    }"]
            # Per entry: the one-source tables (no bbtab_rel2) read source, sign and
            # value; tables with interpolated entries read the second relative
            # source and coefficient with them, all five loads issued together (bit
            # 31 of bbtab_rel2 flags the entries that have a second source; the
            # others repeat their first), so no load waits on another.
            tb_sub += ["    if (bits & 0x80000000u) {",
                       "      using CC = typename Codec<S>::C;",
                       "      const uint32_t tb = tbits[lcell], tbase = tbase_l[lcell];"]
            for two in (True, False):
                tb_sub += ["      if (%sa.bbtab_rel2) {" % ("" if two else "!")]
                for k in range(ns):
                    if ksym[k] == k:
                        continue
                    bit = 1 << k
                    tb_sub += ["        if (tb & %du) {" % bit,
                               "          const uint32_t e_ = tbase + (uint32_t)__builtin_popcount(tb & %du);" % (bit - 1),
                               "          const uint32_t rel = a.bbtab_rel[e_];"]
                    if two:
                        tb_sub += ["          const uint32_t rel2 = a.bbtab_rel2[e_];",
                                   "          const CC c2_ = a.bbtab_c2[e_];"]
                    tb_sub += ["          const CC sg_ = a.bbtab_sign[e_];",
                               "          const CC rh_ = a.bbtab_rhs[e_];",
                               "          const int ks = (int)(rel & 0xffu), dm = (int)((rel >> 8) & 0xffu) - 128,",
                               "                    di = (int)((rel >> 16) & 0xffu) - 128;",
                               "          CC r_ = sg_ * Codec<S>::decode_dev(cur[ks * RC + lcell + dm * RI + di], (CC)0);"]
                    if two:
                        tb_sub += ["          if (rel2 & 0x80000000u) {",
                                   "            const int ks2 = (int)(rel2 & 0xffu), dm2 = (int)((rel2 >> 8) & 0xffu) - 128,",
                                   "                      di2 = (int)((rel2 >> 16) & 0xffu) - 128;",
                                   "            r_ = r_ + c2_ * Codec<S>::decode_dev(cur[ks2 * RC + lcell + dm2 * RI + di2], (CC)0);",
                                   "          }"]
                    tb_sub += ["          r_ += rh_;",
                               "          L%d[0] = Codec<S>::encode(r_, (CC)0);" % k,
                               "        }"]
                tb_sub += ["      }"]
            tb_sub += ["    }", "  }", "}"]
        tb_kernel = _TB_KERNEL % dict(
            tb_mask=_indent(tb_mask, 8), tb_collect=_indent(tb_collect, 6), tb_entries=_indent(tb_entries), tb_apply=_indent(tb_apply, 4),
            tb_loads=_indent(tb_loads, 6), tb_sub=_indent(tb_sub, 6),
            tb_gdecl=_indent(["S %s;" % ", ".join("G%d[1]" % k for k in range(ns))], 6),
            tb_coords=_indent(coords, 6), tb_decode=_indent(decode, 6), tb_collide=_indent(collide, 6),
            tb_lds_stores=_indent(["nxt[%d * RC + lcell] = G%d[0];" % (k, k) for k in range(ns)], 6))
        tb_launch = _TB_LAUNCH % {}
    else:
        tb_kernel = ""
        tb_launch = _TB_LAUNCH_NONE
        # up to D3Q19: what a thread holds of more populations does not fit its registers
        if ns <= 19 and not rel and all(abs(c) <= 1 for v in vel for c in v):
            tb_launch = _PAIR_LAUNCH % {} + _TB_LAUNCH_NONE
            tb_kernel = _pair_source(vel, ksym, decode, coords, collide)
    return _TEMPLATE % dict(
        tb_kernel=tb_kernel, tb_launch=tb_launch, pair_ok=int(dim == 3 and bool(tb_kernel)), unit_vel=int(all(abs(c) <= 1 for v in vel for c in v)),
        hash=spec_hash(spec), ns=ns, nc=spec.nconsm, dim=dim, paired=bool(sig_f2m),
        vel=vel_txt,
        loads=_indent(loads), bbsub=_indent(bbsub), bbsub_ok=int(ksym is not None),
        gdecl=_indent(gdecl), coords=_indent(coords, 4), decode=_indent(decode, 4), vstores=_indent(vstores),
        collide=_indent(collide, 2),
        f2m_loads=_indent(f2m_loads), f2m_full=_indent(f2m_full), f2m_stores=_indent(f2m_stores),
        m2f_loads=_indent(m2f_loads), m2f_full=_indent(m2f_full), m2f_stores=_indent(m2f_stores),
        eq_loads=_indent(eq_loads), eq_body=_indent(eq_body), eq_stores=_indent(eq_stores),
        rx_loads=_indent(rx_loads), rx_body=_indent(rx_body), rx_stores=_indent(rx_stores),
        st_coords=_indent(coords), st_loads=_indent(st_loads), st_body=_indent(st_body),
        st_stores=_indent(st_stores),
        eqm2f_loads=_indent(eqm2f_loads), eqm2f_opaque=_indent(eqm2f_opaque),
    )
