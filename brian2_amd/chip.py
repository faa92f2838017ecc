"""A network without delays over the whole chip, many steps in a launch.

Networks of one group with synapses onto itself whose events carry no more than their number
(resident.plain_network), too large or too heavy for the one workgroup of resident.py: a
workgroup has 64 neurons, whose state its registers hold through all steps of the launch, and
what the workgroups tell each other after a step is one word of spikes each.
"""
import re

from .codegen import ParamStruct, source_header
from .kernels import chain_lines, group_block, group_statements, identifiers, split_update

SPINS = 1 << 22  # polls of the others' words before a launch gives up (seconds)
LATE = 32  # status of a launch that changed nothing, as not all its workgroups came to run


HERE = 3  # words behind the exchange's: workgroups that run (bit 32: one has given up), workgroups
#           waited for beside the launch's own, polls already made


def here_at(words):
    """Place of the HERE words behind so many words of an exchange (in a cache line of their own)."""
    return -(-words // 64) * 64


def arrival_function(words, grid):
    """hb_all_here(xch, status): whether all workgroups of the launch run.  If not, it ends before it
    has changed anything.

    A kernel of another stream may hold the compute units that some of them need; the others, which
    wait, then give up.  They agree on it: who gives up marks the count that it last saw, which
    fails if the count has changed, and a complete count is never marked.  Status 32: the launch can
    be made again.  Once all run, every later wait ends.

    The kernel arrives (arrive_line) first of all and asks behind its loads: 4000 COBAHH neurons
    121 us for 2 steps, as without it; arriving and asking at once 134.  A function of its own, with
    its constants in memory: as part of the kernel its scalars take registers from the steps (5.20
    us each instead of 5.08)."""
    return f"""
__device__ __attribute__((noinline)) int hb_all_here(unsigned long long* xch, int* status) {{
    unsigned long long* const here = xch + {here_at(words)};
    const unsigned long long late = 1ull << 32;
    const int all = {grid} + (int)here[1];
    unsigned long long x = __hip_atomic_load(here, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int spin = (int)here[2]; !(x & late) && (int)x < all; spin++) {{
        if (spin >= {SPINS}) {{
            const unsigned long long y = atomicCAS(here, x, x | late);
            x = y == x ? x | late : y;
        }} else {{
            x = __hip_atomic_load(here, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }}
    }}
    if (x & late) atomicOr(status, {LATE});
    return x & late ? 0 : 1;
}}"""


def arrive_line(words):
    return (f"    if (threadIdx.x == 0) (void)__hip_atomic_fetch_add(p.xch + {here_at(words)}, 1ull, __ATOMIC_RELAXED, "
            "__HIP_MEMORY_SCOPE_AGENT);")


ARRIVAL = [
    "    {",
    "        __shared__ int s_here;",
    "        if (threadIdx.x == 0) s_here = hb_all_here(p.xch, p.status);",
    "        __syncthreads();",
    "        if (__builtin_amdgcn_readfirstlane(s_here) == 0) return;  // (a scalar)",
    "    }",
]


def monitor_fields(ps, g):
    """Fields of a group's monitors."""
    if g.smon:
        ps.ptr("mon_i", "int")
        ps.ptr("mon_step", "int")
        ps.ptr("mon_n", "unsigned long long")
        ps.ptr("mon_count", "int")
        ps.val("mon_cap", "long long")
        ps.val("mon_start", "int")
        ps.val("mon_stop", "int")
    if g.rmon:
        ps.ptr("rate_cnt", "int")
        ps.val("rate_row0", "long long")
        ps.val("rate_rows", "long long")
        ps.val("rate_start", "int")
        ps.val("rate_stop", "int")
    if g.stmon:
        ps.ptr("rec_idx", "int", const=True)
        ps.ptr("rec_buf", "double")
        ps.val("rec_row0", "long long")
        ps.val("rec_rows", "long long")
        ps.val("n_rec", "int")
        ps.val("pad_rec", "int")


def place_lines(first):
    """The place of neuron i among the recorded ones (hb_rec, -1: not recorded)."""
    return [
        "int hb_rec = -1;",
        f"if ({first}) {{",
        "    int lo = 0, hi = p.n_rec;",
        "    while (lo < hi) { const int m = (lo + hi) >> 1; if (p.rec_idx[m] < i) lo = m + 1; else hi = m; }",
        "    if (lo < p.n_rec && p.rec_idx[lo] == i) hb_rec = lo;",
        "}",
    ]


def record_lines(g, first, row, was={}):
    """The recorded variables' values to row `row`, by the threads for which `first` holds
    (was: {variable: what holds its value at that point})."""
    nv = len(g.stmon.variables)
    return [f"if ({first} && hb_rec >= 0 && {row} >= 0 && {row} < p.rec_rows) {{",
            f"    double* const o_ = p.rec_buf + (size_t)({row}) * {nv} * p.n_rec + hb_rec;"] + [
        f"    o_[(size_t){a} * p.n_rec] = (double){was.get(v, v)};" for a, v in enumerate(g.stmon.variables)] + ["}"]


class ChipSteps:
    """Source of the kernel (a workgroup per 64 neurons; all of them have to run at once).

    A step's word goes into the exchange as two 8-byte atomics, each a half of the word and the
    step's number: what is read is complete or not there yet, so neither fences nor a counter are
    needed (a barrier with fences of 63 workgroups takes 4.7 us, one with a counter 2.1).  There
    are two places per workgroup in turn: who writes step s + 2 has read everybody's s + 1, which
    they write when they have read s.  The words' set bits become a list of sources in LDS; a
    lane per source loads the word of this workgroup's 64 targets from the source's row of the
    pathway's bit matrix; a neuron's events are counted bit by bit, with the words in scalar
    registers, and applied pathway by pathway.

    waves: an update's independent heavy parts (kernels.split_update) have a wave each, which
    hands its results to the others through LDS; all else every wave does alike, so that each
    has the state.  An update of many exponentials is bound by the instructions that one wave
    issues, and the other SIMDs would be idle.

    What bounds it: the chain words -> rows -> update -> words.  4000 COBAHH neurons, us per
    step: 36.8 as three launches that stage the events (29.2 with functions without branches),
    12.8 as one launch a step that counts its events itself, 8.6 with the update's parts on
    waves, 6.4 with all steps in a cooperative launch, 5.7 in an ordinary one.

    group, scalars {(tag, name): (value, ctype)}; pathways [(variable, operator, C expression
    of the operand, first source, sources)]; consts [(field, C type)] of the operands'
    constants; mode: when a reset happens ('fused': at once, 'deferred': after the events)"""

    def __init__(self, group, scalars, pathways, consts, n_words, mode):
        g = self.group = group
        self.scalars, self.pathways, self.n_words = scalars, list(pathways), int(n_words)
        NW, R = self.n_words, len(self.pathways)
        C = -(-NW // 64)
        parts = split_update(g.su, 4)
        parts = parts if len(parts) > 1 else []
        W = self.waves = max(1, len(parts))
        ps = ParamStruct(f"hbc_{g.name}")
        ps.val("step0", "long long")
        ps.val("dt", "double")
        ps.val("n_steps", "int")
        ps.val("N", "int")
        for v, ct in g.vars.items():
            ps.ptr(f"a_{v}", "unsigned char" if ct == "bool" else ct)
        for (tg, n), (_, ct) in sorted(scalars.items()):
            ps.val(f"{tg}_{n}", ct)
        for n, ct in consts:
            ps.val(n, ct)
        for r in range(R):
            ps.ptr(f"bits{r}", "unsigned long long", const=True)  # [sources][n_words]
            ps.ptr(f"events{r}", "unsigned long long")  # per workgroup
        ps.ptr("xch", "unsigned long long")  # [2][n_words][2]
        ps.ptr("status", "int")
        monitor_fields(ps, g)
        self.struct = ps
        self.kernel_name = f"chip_{g.name}"

        def block(tag, spec, extra=()):
            return group_block(tag, spec, g.vars, scalars, g.float_t, extra)

        first = "threadIdx.x < 64"
        k = [source_header(64 * W), ps.c_decl(), arrival_function(4 * NW, NW)]
        k.append(f'extern "C" __global__ void __launch_bounds__({64 * W}) {self.kernel_name}(const {ps.name} p) {{')
        k += [
            arrive_line(4 * NW),
            "    const int hb_lane = threadIdx.x & 63, hb_blk = blockIdx.x;",
            "    const int hb_wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);",
            "    const int i = hb_blk * 64 + hb_lane, N = p.N, _idx = i;",
            "    const bool hb_act = i < N;",
            "    const double dt = p.dt;",
            "    (void)_idx; (void)hb_wave; (void)dt;",
            "    __shared__ unsigned short s_src[4096];",
            f"    __shared__ unsigned int s_cnt[2][{R}][64];",
            "    __shared__ int s_late[2];",
        ]
        sts = group_statements("su", g.su, g.vars, scalars, g.float_t)
        done = {x for w in parts for x in w}
        read = set().union(*(identifiers([st]) for x, (st, _) in enumerate(sts) if x not in done), set())
        handed = sorted(x for x in done if sts[x][0]["var"] in read)
        for x in handed:
            ct = re.match(r"(?:const )?(\w+(?: long)?) ", sts[x][1][0]).group(1)
            k.append(f"    __shared__ {ct} s_part_{sts[x][0]['var']}[2][64];")
        for v, ct in g.vars.items():
            k.append(f"    {ct} {v} = hb_act ? p.a_{v}[i]{' != 0' if ct == 'bool' else ''} : ({ct})0;")
            if ct != "bool":
                k.append(f'    asm volatile("" : "+v"({v}));  // waited for here, not in the loop behind its stores')
        k += [
            f"    unsigned int hb_e[{R}];",
            f"    for (int r = 0; r < {R}; r++) hb_e[r] = 0u;",
            "    bool hb_cond = false, hb_ok = true;",
        ]
        if g.stmon:
            k += ["    " + x for x in place_lines("hb_act")]

        # events of the step whose number from the launch's start, plus one, is tag
        k += [
            f"    auto hb_pull = [&](const unsigned int tag, unsigned int (&n)[{R}]) {{",
            f"        const unsigned long long* const x = p.xch + (size_t)(tag & 1u) * {2 * NW};",
            f"        unsigned long long lo[{C}], hi[{C}];",
            "        for (int spin = 0;; spin++) {",
            "            bool there = true;",
            "            #pragma unroll",
            f"            for (int c = 0; c < {C}; c++) {{",
            f"                const int w = c * 64 + hb_lane < {NW} ? c * 64 + hb_lane : {NW - 1};",
            "                lo[c] = __hip_atomic_load(x + 2 * w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);",
            "                hi[c] = __hip_atomic_load(x + 2 * w + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);",
            "            }",
            "            #pragma unroll",
            f"            for (int c = 0; c < {C}; c++)",
            "                there = there && (unsigned int)(lo[c] >> 32) == tag && (unsigned int)(hi[c] >> 32) == tag;",
            "            if (__builtin_amdgcn_ballot_w64(!there) == 0ull) break;",
            f"            if (spin == {SPINS}) {{ hb_ok = false; if (hb_lane == 0) atomicOr(p.status, 16); break; }}",
            "        }",
            f"        for (int r = 0; r < {R}; r++) n[r] = 0u;",
            "        #pragma unroll",
            f"        for (int c = 0; c < {C}; c++) {{",
            f"            unsigned long long w = c * 64 + hb_lane < {NW} && hb_ok ? hi[c] << 32 | (unsigned int)lo[c] : 0ull;",
            "            if (__builtin_amdgcn_ballot_w64(w != 0ull) == 0ull) continue;",
            "            // the chunk's sources, in order (this wave's own list: its accesses stay in order)",
            "            const int in_ = hb_wave_incl_scan(__popcll(w));",
            "            const int m = __builtin_amdgcn_readlane(in_, 63);",
            "            for (int o = in_ - __popcll(w); w; w &= w - 1ull) s_src[o++] = (unsigned short)(hb_lane << 6 | __builtin_ctzll(w));",
            "            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, \"wavefront\");",
            "            for (int s0 = 0; s0 < m; s0 += 64) {",
            "                const int src = s0 + hb_lane < m ? c * 4096 + (int)s_src[s0 + hb_lane < m ? s0 + hb_lane : 0] : -1;",
        ]
        for r, (_, _, _, a, cnt) in enumerate(self.pathways):
            k += [
                f"                const bool ok{r} = (unsigned int)(src - {a}) < {cnt}u;",
                f"                const unsigned long long x{r} = p.bits{r}[ok{r} ? (size_t)(src - {a}) * {NW} + hb_blk : (size_t)0];",
            ]
        for r in range(R):
            k += [
                "                {",
                f"                    const unsigned long long x = ok{r} ? x{r} : 0ull;",
                f"                    hb_e[{r}] += (unsigned int)__popcll(x);",
                "                    for (unsigned long long m = __builtin_amdgcn_ballot_w64(x != 0ull); m; m &= m - 1ull) {",
                "                        const int l = __builtin_ctzll(m);",
                "                        const unsigned int lo_ = (unsigned int)__builtin_amdgcn_readlane((int)x, l);",
                "                        const unsigned int hi_ = (unsigned int)__builtin_amdgcn_readlane((int)(x >> 32), l);",
                f"                        n[{r}] += ((hb_lane < 32 ? lo_ : hi_) >> (hb_lane & 31)) & 1u;",
                "                    }",
                "                }",
            ]
        k += [
            "            }",
            "            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, \"wavefront\");",
            "        }",
            "    };",
            "    // the events of the step before step hb_s of the launch, applied (hb_ok: no workgroup missing)",
            "    auto hb_events = [&](const int hb_s) {",
            f"        unsigned int hb_n[{R}];",
        ]
        if W > 1:
            k += [
                "        if (hb_wave == 0) {",
                "            hb_pull((unsigned int)hb_s, hb_n);",
                "            #pragma unroll",
                f"            for (int r = 0; r < {R}; r++) s_cnt[hb_s & 1][r][hb_lane] = hb_n[r];",
                "            if (hb_lane == 0) s_late[hb_s & 1] = hb_ok ? 0 : 1;",
                "        }",
                "        __syncthreads();",
                "        #pragma unroll",
                f"        for (int r = 0; r < {R}; r++) hb_n[r] = s_cnt[hb_s & 1][r][hb_lane];",
                "        hb_ok = s_late[hb_s & 1] == 0;",
            ]
        else:
            k.append("        hb_pull((unsigned int)hb_s, hb_n);")
        for r, (var, op, val, _, _) in enumerate(self.pathways):
            k.append(f"        for (unsigned int n_ = hb_n[{r}]; n_ > 0u; n_--) {var} {op} {val};")
        if mode == "deferred":
            k += ["        if (hb_cond) { // reset of the step before, after its propagation, at its time",
                  "            const double t = (double)(p.step0 + hb_s - 1) * dt;", "            (void)t;"]
            k += ["            " + x for x in block("rs", g.rs)] + ["        }"]
        k += ["    };"] + ARRIVAL + ["    for (int hb_s = 0; hb_s < p.n_steps; hb_s++) {", "        const long long hb_step = p.step0 + hb_s;",
              "        const double t = (double)hb_step * dt;", "        (void)t;",
              "        if (hb_s > 0) { hb_events(hb_s); if (!hb_ok) return; }"]
        if g.stmon:
            row = "(hb_step - p.rec_row0)" if g.stmon.when == "start" else "(hb_step - 1 - p.rec_row0)"
            k += ["        " + x for x in record_lines(g, first, row)]
        for w, part in enumerate(parts):
            k.append(f"        {'else ' if w else ''}if (hb_wave == {w}) {{")
            for x in part:
                k += ["            " + y for y in sts[x][1]]
                if x in handed:
                    k.append(f"            s_part_{sts[x][0]['var']}[hb_s & 1][hb_lane] = {sts[x][0]['var']};")
            k.append("        }")
        if W > 1:
            k.append("        __syncthreads();  // (two sets of results in turn: one barrier is enough)")
        k += ["        hb_cond = false;", "        {"]
        for x, (st, ls) in enumerate(sts):
            if x not in done:
                k += ["            " + y for y in ls]
            elif x in handed:
                k.append(f"            const auto {st['var']} = s_part_{st['var']}[hb_s & 1][hb_lane];")
        k.append("        }")
        if g.th is not None:
            k += ["        {"] + ["            " + x for x in block("th", g.th, {"_cond": "bool"})]
            k += ["            hb_cond = _cond && hb_act;", "        }"]
            if g.uses_refractory:
                k.append("        if (hb_cond) { not_refractory = false; lastspike = t; }")
        if mode == "fused":
            k += ["        if (hb_cond) {"] + ["            " + x for x in block("rs", g.rs)] + ["        }"]
        k += [
            "        const unsigned long long hb_w = __builtin_amdgcn_ballot_w64(hb_cond);",
            f"        if ({first}) {{",
            "            if (hb_lane < 2) {  // first of all: the others wait for it",
            "                const unsigned long long x = hb_lane == 0 ? hb_w & 0xffffffffull : hb_w >> 32;",
            f"                __hip_atomic_store(p.xch + ((size_t)((hb_s + 1) & 1) * {NW} + hb_blk) * 2 + hb_lane,",
            "                                   (unsigned long long)(hb_s + 1) << 32 | x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);",
            "            }",
        ]
        if g.smon:
            k += [
                "            const bool in_ = hb_cond && i >= p.mon_start && i < p.mon_stop;",
                "            const unsigned long long m_ = __builtin_amdgcn_ballot_w64(in_);",
                "            if (m_ != 0ull) {",
                "                unsigned long long o_ = 0ull;",
                "                if (hb_lane == 0) {",
                "                    o_ = atomicAdd(p.mon_n, (unsigned long long)__popcll(m_));",
                "                    if (o_ + (unsigned long long)__popcll(m_) > (unsigned long long)p.mon_cap) atomicOr(p.status, 2);",
                "                }",
                "                o_ = __shfl(o_, 0, 64) + (unsigned long long)__popcll(m_ & ((1ull << hb_lane) - 1ull));",
                "                if (in_ && o_ < (unsigned long long)p.mon_cap) { p.mon_i[o_] = i; p.mon_step[o_] = (int)hb_step; }",
                "                if (in_) p.mon_count[i - p.mon_start] += 1;",
                "            }",
            ]
        if g.rmon:
            k += [
                "            const int c_ = __popcll(__builtin_amdgcn_ballot_w64(hb_cond && i >= p.rate_start && i < p.rate_stop));",
                "            if (hb_lane == 0 && c_ && p.rate_cnt && hb_step - p.rate_row0 >= 0 && hb_step - p.rate_row0 < p.rate_rows)",
                "                atomicAdd(&p.rate_cnt[hb_step - p.rate_row0], c_);",
            ]
        k += [
            "        }",
            "    }",
            "    {  // the last step's events, and the state back to memory",
            "        const long long hb_step = p.step0 + p.n_steps;",
            "        hb_events(p.n_steps);",
            "        (void)hb_step;",
            "        if (!hb_ok) return;",
        ]
        if g.stmon and g.stmon.when == "end":
            k += ["        " + x for x in record_lines(g, first, "(hb_step - 1 - p.rec_row0)")]
        k += ["    }", f"    if ({first}) {{", "        if (hb_act) {"]
        for v, ct in g.vars.items():
            k.append(f"            p.a_{v}[i] = {v}{' ? 1 : 0' if ct == 'bool' else ''};")
        k.append("        }")
        for r in range(R):
            k += [f"        const int e{r} = __builtin_amdgcn_readlane(hb_wave_incl_scan((int)hb_e[{r}]), 63);",
                  f"        if (hb_lane == 0) p.events{r}[hb_blk] += (unsigned long long)e{r};"]
        k += ["    }", "}"]
        self.source = "\n".join(k) + "\n"


class SumSteps:
    """Source of the kernel for a group whose only synapses are a summed variable of itself
    (kernels.OwnSum for larger groups): a wave per neuron, all steps in a launch.

    As in ChipSteps, what the workgroups tell each other goes through memory in 8-byte atomics
    tagged with the step: here the values of the variables that the sum reads of its sources.
    Each workgroup gathers all of them in LDS; a wave's lanes evaluate its neuron's synapses
    (kept in registers where they fit) and the wave adds them up in order; all lanes do the
    neuron's step alike.

    What bounds it: the exchange (2.6 us: a read of all values takes 0.8 and is done three times
    before all are there) and the chain of additions, whose order is the result (300: 1.8 us)."""

    CHUNK = 512
    WAVES = 4  # neurons of a workgroup: 300 neurons 6.0 / 5.6 / 5.9 / 8.4 us per step with 2 / 4 / 8 / 16
    WORDS = 768

    @classmethod
    def takes(cls, n, types):
        """Whether a group of n neurons, whose sum reads variables of these types of its sources,
        is stepped this way: with few values to exchange, as everyone reads them all (and, where
        the sum reads none, with as few workgroups, which run all at once).

        us per step all-to-all against a launch each, fp64 / fp32 (two words or one per neuron):
        50 neurons 3.4 against 4.4 / 2.3 against 4.2, 150 4.1 against 5.5 / 3.3 against 5.0, 300
        5.6 against 5.9 / 4.4 against 5.5, 500 7.5 against 7.2 / 5.7 against 6.9, 1000 13.4
        against 11.0 / 10.2 against 10.1."""
        return n * max(1, sum(2 if ct == "double" else 1 for ct in types)) <= cls.WORDS

    def __init__(self, group, scalars, own, max_degree):
        g = self.group = group
        self.scalars, self.own = scalars, own
        T, CH, W = 64 * self.WAVES, self.CHUNK, self.WAVES
        self.grid = -(-g.N // W)
        kept = max_degree <= CH
        words = [(v, h) for v in own.shared for h in ((0, 1) if g.vars[v] == "double" else (0,))]
        self.n_words = len(words)
        K = -(-g.N // T)  # neurons whose values a thread gathers
        U = CH // 64
        ps = ParamStruct(f"hbw_{g.name}")
        ps.val("step0", "long long")
        ps.val("dt", "double")
        ps.val("n_steps", "int")
        ps.val("N", "int")
        for v, ct in g.vars.items():
            ps.ptr(f"a_{v}", "unsigned char" if ct == "bool" else ct)
        for (tg, n), (_, ct) in sorted(scalars.items()):
            ps.val(f"{tg}_{n}", ct)
        own.fields(ps)  # (z_x_<variable>: the values when the launch begins)
        ps.ptr("xch", "unsigned long long")  # [2][words][N]
        ps.ptr("status", "int")
        monitor_fields(ps, g)
        self.struct = ps
        self.kernel_name = f"sums_{g.name}"

        def block(tag, spec, extra=()):
            return group_block(tag, spec, g.vars, scalars, g.float_t, extra)

        first = "hb_lane == 0"
        k = [source_header(T), ps.c_decl(), arrival_function(2 * len(words) * g.N, self.grid)]
        k.append(f'extern "C" __global__ void __launch_bounds__({T}) {self.kernel_name}(const {ps.name} p) {{')
        k += [
            arrive_line(2 * len(words) * g.N),
            "    const int hb_lane = threadIdx.x & 63;",
            "    const int hb_wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);",
            f"    const int i = (int)blockIdx.x * {W} + hb_wave, N = p.N, _idx = i;  // the same for the wave",
            "    const bool hb_act = i < N;",
            "    const double dt = p.dt;",
            "    (void)_idx; (void)dt;",
            f"    __shared__ __align__(16) {own.vt} s_sum[{W}][{CH}];",
        ] + [f"    __shared__ {g.vars[v]} s_x_{v}[2][{g.N}];" for v in own.shared]
        k += ["    __shared__ int s_late[2];", "    if (threadIdx.x < 2) s_late[threadIdx.x] = 0;", "    __syncthreads();"]
        for v, ct in g.vars.items():
            k.append(f"    {ct} {v} = hb_act ? p.a_{v}[i]{' != 0' if ct == 'bool' else ''} : ({ct})0;")
            if ct != "bool":
                k.append(f'    asm volatile("" : "+v"({v}));  // waited for here, not in the loop behind its stores')
        k += [
            f"    const bool hb_sums = hb_act && i >= {own.t0} && i < {own.t1};",
            "    const unsigned int hb_lo = hb_sums ? p.z_post_ptr[i] : 0u, hb_hi = hb_sums ? p.z_post_ptr[i + 1] : 0u;",
            "    bool hb_cond = false;",
        ]
        sl = [f"{ct} hb_s_{v}[{U}];" for v, ct in own.syn_arrays.items()] + [f"int hb_p[{U}];"]
        ld = ["#pragma unroll", f"for (int hb_u = 0; hb_u < {U}; hb_u++) {{",
              "    const unsigned int q_ = hb_c + hb_u * 64u + hb_lane, k_ = q_ < hb_hi ? q_ : hb_hi - 1u;"]
        ld += [f"    hb_s_{v}[hb_u] = p.z_s_{v}[k_];" for v in own.syn_arrays] + ["    hb_p[hb_u] = p.z_post_pre[k_];", "}"]
        if kept:
            k += ["    " + x for x in sl]
            k += ["    if (hb_hi > hb_lo) {", "        const unsigned int hb_c = hb_lo;"] + ["        " + x for x in ld] + ["    }"]
        if g.stmon:
            k += ["    " + x for x in place_lines("hb_act")]
        k += ARRIVAL + [
            "    for (int hb_s = 0; hb_s < p.n_steps; hb_s++) {",
            "        const long long hb_step = p.step0 + hb_s;",
            "        const double t = (double)hb_step * dt;",
            "        (void)t;",
            "        // the sources' values: of the launch's beginning, or of the step before",
            "        if (hb_s == 0) {",
            f"            for (int x = threadIdx.x; x < {g.N}; x += {T}) {{",
        ] + [f"                s_x_{v}[0][x] = p.z_x_{v}[x];" for v in own.shared] + [
            "            }",
            "        } else {",
            f"            const unsigned long long* const x = p.xch + (size_t)(hb_s & 1) * {len(words) * g.N};",
            f"            unsigned long long hb_v[{K}][{len(words)}];",
            "            for (int spin = 0;; spin++) {",
            "                bool there = true;",
            "                #pragma unroll",
            f"                for (int c = 0; c < {K}; c++) {{",
            f"                    const int j = c * {T} + (int)threadIdx.x < {g.N} ? c * {T} + (int)threadIdx.x : {g.N - 1};",
            "                    #pragma unroll",
            f"                    for (int h = 0; h < {len(words)}; h++) {{",
            f"                        hb_v[c][h] = __hip_atomic_load(x + h * {g.N} + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);",
            "                    }",
            "                }",
            "                #pragma unroll",
            f"                for (int c = 0; c < {K}; c++)",
            "                    #pragma unroll",
            f"                    for (int h = 0; h < {len(words)}; h++) there = there && (int)(hb_v[c][h] >> 32) == hb_s;",
            "                if (__builtin_amdgcn_ballot_w64(!there) == 0ull) break;",
            f"                if (spin == {SPINS}) {{ if (hb_lane == 0) {{ s_late[hb_s & 1] = 1; atomicOr(p.status, 16); }} break; }}",
            "            }",
            "            #pragma unroll",
            f"            for (int c = 0; c < {K}; c++) {{",
            f"                const int j = c * {T} + (int)threadIdx.x;",
            f"                if (j < {g.N}) {{",
        ]
        at = {x: n for n, x in enumerate(words)}
        for v in own.shared:
            if g.vars[v] == "double":
                k.append(f"                    s_x_{v}[hb_s & 1][j] = __builtin_bit_cast(double, hb_v[c][{at[(v, 1)]}] << 32 | "
                         f"(unsigned int)hb_v[c][{at[(v, 0)]}]);")
            else:
                k.append(f"                    s_x_{v}[hb_s & 1][j] = __builtin_bit_cast(float, (unsigned int)hb_v[c][{at[(v, 0)]}]);")
        k += [
            "                }",
            "            }",
            "        }",
            "        __syncthreads();  // (two sets of values in turn: one barrier is enough)",
            "        if (s_late[hb_s & 1] != 0) return;",
            f"        const {own.target_t} hb_was = {own.target};  // before this step's sum",
            "        (void)hb_was;",
            "        if (hb_sums) {",
            f"            {own.target_t} hb_acc = ({own.target_t})0;",
            f"            for (unsigned int hb_c = hb_lo; hb_c < hb_hi; hb_c += {CH}u) {{",
        ]
        if not kept:
            k += ["                " + x for x in sl + ld]
        k += ["                #pragma unroll", f"                for (int hb_u = 0; hb_u < {U}; hb_u++) {{",
              "                    const int _presynaptic_idx = hb_p[hb_u], _postsynaptic_idx = i;",
              "                    (void)_presynaptic_idx; (void)_postsynaptic_idx;"]
        k += [f"                    const {ct} {v} = hb_s_{v}[hb_u];" for v, ct in own.syn_arrays.items()]
        k += [f"                    const {own.var_types[n]} {n} = s_x_{v}[hb_s & 1][_presynaptic_idx];"
              for n, v in sorted(own.pre_reads.items())]
        k += [f"                    const {own.var_types[n]} {n} = {v};" for n, v in sorted(own.post_reads.items())]
        k += ["                    " + x for x in own.code]
        k += [
            "                    // past the end -0.0, which changes no sum",
            f"                    s_sum[hb_wave][hb_u * 64 + hb_lane] = hb_c + hb_u * 64u + hb_lane < hb_hi ? _synaptic_var : ({own.vt})-0.0;",
            "                }",
        ]
        k += ["                " + x for x in chain_lines(CH, own.vt, "hb_wave", f"(hb_hi - hb_c < {CH}u ? hb_hi - hb_c : {CH}u)")]
        k += ["            }", f"            {own.target} = hb_acc;", "        }"]
        if g.stmon:
            row = "(hb_step - p.rec_row0)" if g.stmon.when == "start" else "(hb_step - 1 - p.rec_row0)"
            k += ["        " + x for x in record_lines(g, first, row, {own.target: "hb_was"})]
        k += ["        hb_cond = false;", "        {"] + ["            " + x for x in block("su", g.su)] + ["        }"]
        if g.th is not None:
            k += ["        {"] + ["            " + x for x in block("th", g.th, {"_cond": "bool"})]
            k += ["            hb_cond = _cond && hb_act;", "        }"]
            if g.uses_refractory:
                k.append("        if (hb_cond) { not_refractory = false; lastspike = t; }")
        if g.rs is not None:
            k += ["        if (hb_cond) {"] + ["            " + x for x in block("rs", g.rs)] + ["        }"]
        k += ["        if (hb_lane == 0 && hb_act) {  // first of all: the others wait for it",
              f"            unsigned long long* const hb_o = p.xch + (size_t)((hb_s + 1) & 1) * {len(words) * g.N} + i;",
              "            const unsigned long long hb_tag = (unsigned long long)(hb_s + 1) << 32;"]
        for n, (v, h) in enumerate(words):
            if g.vars[v] == "double":
                bits = f"(__builtin_bit_cast(unsigned long long, {v}) {'>> 32' if h else '& 0xffffffffull'})"
            else:
                bits = f"__builtin_bit_cast(unsigned int, {v})"
            k.append(f"            __hip_atomic_store(hb_o + {n * g.N}, hb_tag | {bits}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);")
        if g.smon:
            k += [
                "            if (hb_cond && i >= p.mon_start && i < p.mon_stop) {",
                "                const unsigned long long o_ = atomicAdd(p.mon_n, 1ull);",
                "                if (o_ < (unsigned long long)p.mon_cap) { p.mon_i[o_] = i; p.mon_step[o_] = (int)hb_step; }",
                "                else atomicOr(p.status, 2);",
                "                p.mon_count[i - p.mon_start] += 1;",
                "            }",
            ]
        if g.rmon:
            k += [
                "            if (hb_cond && i >= p.rate_start && i < p.rate_stop && p.rate_cnt && hb_step - p.rate_row0 >= 0 && "
                "hb_step - p.rate_row0 < p.rate_rows)",
                "                atomicAdd(&p.rate_cnt[hb_step - p.rate_row0], 1);",
            ]
        k += ["        }", "    }"]
        if g.stmon and g.stmon.when == "end":
            k += ["    {", "        const long long hb_step = p.step0 + p.n_steps;"]
            k += ["        " + x for x in record_lines(g, first, "(hb_step - 1 - p.rec_row0)")] + ["    }"]
        k += ["    if (hb_lane == 0 && hb_act) {"]
        for v, ct in g.vars.items():
            k.append(f"        p.a_{v}[i] = {v}{' ? 1 : 0' if ct == 'bool' else ''};")
        k += ["    }", "}"]
        self.source = "\n".join(k) + "\n"
