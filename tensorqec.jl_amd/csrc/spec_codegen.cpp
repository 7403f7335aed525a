// spec_codegen.cpp — see spec_codegen.hpp.
//
// The generated kernel follows the generic FP32 fused kernel of
// tqec_hip.hip step for step (syndrome staging, per-tensor power-of-two
// scaling with tagged LDS maxima, low-exponent flag, finalisation and FP64
// re-check list), with every descriptor field substituted by its value.
#include "spec_codegen.hpp"

#include <algorithm>
#include <array>
#include <cstdio>
#include <cctype>
#include <cmath>
#include <sstream>
#include <vector>

namespace tqec {

namespace {

size_t round_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

constexpr size_t kCuLds = 160 * 1024;   // of a CU

struct Layout {
    size_t work = 0, tab = 0, mx = 0, ex = 0, syn = 0, low = 0, red = 0, total = 0;
    size_t tab_entries = 0;
};

// x spread onto the given bit positions: bit t of x goes to bits[t].
uint32_t pdep(uint32_t x, const std::vector<int> &bits) {
    uint32_t r = 0;
    for (size_t j = 0; j < bits.size(); ++j) r |= ((x >> j) & 1u) << bits[j];
    return r;
}

// ---- steps with few outputs and a long contraction -----------------------
//
// One lane per output leaves most of a workgroup idle and makes each output a
// serial chain of 2^nk multiply-adds (toric L=5 ends in 64 outputs of 2^18
// terms: 38% of its time).  In the configurations that need not keep the
// generic kernel's order of summation (mfma32), such a step gives every thread
// a block of up to 64 outputs and a share of the contraction: the block's
// operand values are loaded once per k, consecutive threads take consecutive
// k, and the partial sums meet in a shuffle tree and, across waves, in LDS.
// Measured: that step of toric L=5 24.3 -> 3.4 M cycles (its 16.8 MB per
// syndrome at 5.6 TB/s over the chip, the rate of a large copy), 512 syndromes
// 29.2 -> 20.9 ms with the smaller MFMA blocks of emit_outputs_mfma32; the
// circuit-level d=3, 3-round plan 400 -> 358 us per 16,384.

// Output bits held per thread, -1 when the step does not run this way.  The
// block is as large as leaves each thread at least eight terms.
int split_k_block(const StepDesc &st, const SpecCfg &cfg) {
    if (!cfg.mfma32 || cfg.fp64 || cfg.glog != 0 || st.rc > 8 || st.nk < 6) return -1;
    if ((1 << st.rc) > cfg.threads) return -1;
    for (int rb = std::min(st.rc, 6); rb >= 0; --rb)
        if ((int64_t)(cfg.threads >> (st.rc - rb)) * 8 <= (int64_t(1) << st.nk)) return rb;
    return -1;
}

// LDS floats of the partial sums: one per output and wave of its threads.
size_t split_k_entries(const CompiledPlan &cp, const SpecCfg &cfg) {
    size_t n = 0;
    for (const StepDesc &st : cp.steps) {
        const int rb = split_k_block(st, cfg);
        if (rb < 0) continue;
        const int thr = cfg.threads >> (st.rc - rb);   // threads sharing a block
        n = std::max(n, (size_t)std::max(1, thr / 64) << st.rc);
    }
    return n;
}

// ---- slab kernels: the smaller intermediates in LDS ----------------------
//
// A slab plan's steps are bound by memory traffic, and the widest few tensors
// make the slab necessary while most of the traffic is in smaller ones, so as
// many intermediates as fit live in LDS instead, each from the step that makes
// it to the step that reads it.  The LDS of a CU is divided among as many waves
// per SIMD as the configuration asks for, two at least (what a slab kernel's
// registers allow when it is held to none).  Measured with 256 threads and two
// (76 KB): circuit-level d=5, 2 rounds 2.79 -> 2.22 ms per 4,096 (it ran at 4.7
// TB/s of HBM traffic, 34% of it in tensors of at most 2^13 entries), toric L=3
// 772 -> 594 us per 8,192; toric L=5, whose traffic is in its 2^21-entry
// tensors, is unchanged.  With BF16 steps the d=5 plan takes 26.3 ms per 16,384
// instead of 33.5 at two waves; at four, with the LDS divided by two, its tuned
// configuration took 37.3, divided by four 31.0, without placement 33.8.  Fewer
// workgroups with smaller slabs in all (171 MB, less than the memory-side
// cache) changed nothing.
struct Places {
    std::vector<int64_t> lds;                // per step: output's LDS entry offset (per syndrome), -1 in the slab
    std::vector<std::array<int, 2>> prod;    // per step: steps that made its operands, -1 for tables
    int64_t entries = 0;                     // LDS entries per syndrome
};

constexpr size_t kSlabLds = 152 * 1024;      // of 160 KB per CU, the rest for scales and syndromes

Places slab_places(const CompiledPlan &cp, const SpecCfg &cfg) {
    const int ns = (int)cp.steps.size();
    Places P;
    P.lds.assign(ns, -1);
    P.prod.assign(ns, {-1, -1});
    std::vector<int> last(ns, ns);           // step that reads the output (the root: after the last)
    for (int s = 0; s < ns; ++s)
        for (int side = 0; side < 2; ++side) {
            const OperandDesc &op = side ? cp.steps[s].b : cp.steps[s].a;
            if (op.kind != kInter) continue;
            for (int j = s - 1; j >= 0; --j)
                if (cp.steps[j].c_off == op.off) {
                    P.prod[s][side] = j;
                    last[j] = s;
                    break;
                }
        }
    if (!cfg.slab || cfg.fp64) return P;
    const int per_cu = 256 * std::max(2, cfg.waves);   // threads of a CU
    const int64_t room = (int64_t)(kSlabLds * std::min(cfg.threads, per_cu) / per_cu / 4) >> cfg.glog;
    std::vector<int> order(ns);
    for (int s = 0; s < ns; ++s) order[s] = s;
    int64_t best = 0;
    for (int rule = 0; rule < 2; ++rule) {
        // smallest tensors first, or shortest-lived first
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
            const int rx = cp.steps[x].rc, ry = cp.steps[y].rc, lx = last[x] - x, ly = last[y] - y;
            return rule == 0 ? std::make_pair(rx, lx) < std::make_pair(ry, ly) : std::make_pair(lx, -rx) < std::make_pair(ly, -ry);
        });
        std::vector<int64_t> at(ns, -1);
        int64_t placed = 0, top = 0;
        for (int s : order) {
            const int64_t size = int64_t(1) << cp.steps[s].rc;
            // lowest gap between the tensors that live at the same time
            std::vector<std::pair<int64_t, int64_t>> busy;
            for (int j = 0; j < ns; ++j)
                if (at[j] >= 0 && j <= last[s] && s <= last[j]) busy.emplace_back(at[j], at[j] + (int64_t(1) << cp.steps[j].rc));
            std::sort(busy.begin(), busy.end());
            int64_t off = 0;
            for (auto &b : busy) {
                if (off + size <= b.first) break;
                off = std::max(off, b.second);
            }
            if (off + size > room) continue;
            at[s] = off;
            placed += size;
            top = std::max(top, off + size);
        }
        if (placed > best) {
            best = placed;
            P.lds = at;
            P.entries = top;
        }
    }
    return P;
}

Layout layout(const CompiledPlan &cp, const SpecCfg &cfg) {
    const size_t G = size_t(1) << cfg.glog;
    const size_t elem = cfg.fp64 ? 8 : 4;
    Layout L;
    L.tab_entries = cp.const_pool.size() + cp.sliced_pool.size();
    size_t off = 0;
    L.work = off;
    if (!cfg.slab) off += round_up((size_t)std::max<int64_t>(1, cp.ws_entries) * G * elem, 16);
    else off += round_up((size_t)slab_places(cp, cfg).entries * G * elem, 16);
    L.tab = off;
    if (cfg.tab_lds) off += round_up(std::max<size_t>(1, L.tab_entries) * elem, 16);
    L.mx = off;
    if (!cfg.fp64) off += (size_t)std::max(1, cp.n_slots) * G * 8;
    L.ex = off;
    if (!cfg.fp64) off += (size_t)std::max(1, cp.n_slots) * G * 4;
    L.syn = off;
    off += round_up((size_t)std::max(1, cp.n_syn) * G, 4);
    L.low = off;
    if (!cfg.fp64) off += G * 4;
    off = round_up(off, 16);
    L.red = off;
    off += split_k_entries(cp, cfg) * 4;
    L.total = round_up(off, 16);
    return L;
}

// gather_bits(c, op) as an expression of `c`.
std::string gather_expr(const OperandDesc &op) {
    std::ostringstream s;
    bool any = false;
    for (int i = 0; i < op.nseg; ++i) {
        const Seg &g = op.seg[i];
        if (g.width <= 0) continue;
        const unsigned mask = (g.width >= 32) ? 0xffffffffu : ((1u << g.width) - 1u);
        if (any) s << " | ";
        s << "(((c >> " << g.src << ") & " << mask << "u) << " << g.dst << ")";
        any = true;
    }
    if (!any) return "0u";
    return s.str();
}

// Base pointer of an operand (fused_base).
// `lds`: entry offset of an intermediate that a slab kernel keeps in LDS, or -1.
void emit_base(std::ostringstream &o, const char *name, const OperandDesc &op, size_t const_n, int64_t lds) {
    if (op.kind == kInter) {
        o << "    const T *" << name << " = " << (lds >= 0 ? "lwork + " : "work + ")
          << (long long)(lds >= 0 ? lds : op.off) << " * G + g;\n";
    } else if (op.kind == kConst) {
        o << "    const T *" << name << " = tab + " << (long long)op.off << ";\n";
    } else {
        o << "    unsigned v_" << name << " = 0u;\n";
        for (int j = 0; j < op.nev; ++j)
            o << "    v_" << name << " |= (unsigned)synl[" << op.ev_bit[j] << " * G + g] << " << j << ";\n";
        o << "    const T *" << name << " = tab + " << (long long)(const_n + (size_t)op.off) << " + (v_" << name
          << " << " << op.rank << ");\n";
    }
}

// Bits an operand index can take from the output index.
uint32_t gathered_mask(const OperandDesc &op) {
    uint32_t m = 0;
    for (int i = 0; i < op.nseg; ++i) {
        const Seg &g = op.seg[i];
        if (g.width <= 0) continue;
        const uint32_t w = (g.width >= 32) ? 0xffffffffu : ((1u << g.width) - 1u);
        m |= w << g.dst;
    }
    return m;
}

// op_load_sum for element index (idx_var | kconst).  The index is written
// as a sum when the constant's bits cannot meet the gathered bits, which
// lets the compiler fold it into the LDS instruction's offset.
std::string load_expr(const OperandDesc &op, const char *base, const char *idx, uint32_t kconst,
                      std::ostringstream &pre, const std::string &tmp) {
    std::ostringstream s;
    const uint32_t gm = gathered_mask(op);
    uint32_t allk = kconst;
    if (op.kind == kInter)
        for (uint32_t q = 0; q < (1u << op.nsingle); ++q) allk |= kconst | (q << op.sshift);
    const char *join = (gm & allk) ? " | " : " + ";
    if (op.kind != kInter) {
        s << base << "[" << idx << join << kconst << "u]";
        return s.str();
    }
    if (op.nsingle == 0) {
        s << base << "[(" << idx << join << kconst << "u) << GLOG]";
        return s.str();
    }
    // T s = 0; for q: s += base[(idx | q << sshift) * G]
    pre << "        T " << tmp << " = 0;\n";
    const uint32_t ns = 1u << op.nsingle;
    for (uint32_t q = 0; q < ns; ++q)
        pre << "        " << tmp << " += " << base << "[(" << idx << join << (kconst | (q << op.sshift))
            << "u) << GLOG];\n";
    return tmp;
}

// Output bits of a step that feed an operand's index (the segments' sources).
uint32_t source_mask(const OperandDesc &op) {
    uint32_t m = 0;
    for (int i = 0; i < op.nseg; ++i) {
        const Seg &g = op.seg[i];
        if (g.width <= 0) continue;
        const uint32_t w = (g.width >= 32) ? 0xffffffffu : ((1u << g.width) - 1u);
        m |= w << g.src;
    }
    return m;
}

// `expr` with every whole-word `c` replaced by `by`.
std::string subst_c(const std::string &expr, const std::string &by) {
    std::string r;
    for (size_t i = 0; i < expr.size(); ++i) {
        if (expr[i] == 'c' && (i == 0 || !isalnum((unsigned char)expr[i - 1])) &&
            (i + 1 == expr.size() || !isalnum((unsigned char)expr[i + 1])))
            r += "(" + by + ")";
        else
            r += expr[i];
    }
    return r;
}

// The output loop of a step.  Lane c0 (< CSTEP) owns the outputs whose low
// bits are c0.  Up to `block` of them are computed together: the block
// varies output bits that feed only A or only B, so an A row (or B row)
// loaded once serves several outputs (register blocking of the small
// per-syndrome contraction); all loads come before the fma chains and the
// stores after them.  Every output keeps the generic kernel's order of
// operations (k ascending, single-side sums first), so results are
// bit-identical.
// Contraction terms per output unrolled in full; longer contractions run a
// loop over chunks of this many terms (same order of the multiply-adds).
constexpr uint32_t kMaxUnrollK = 16;

void emit_outputs(std::ostringstream &o, const StepDesc &st, int cstep, int block, bool fp64) {
    const OperandDesc &A = st.a, &B = st.b;
    const int rc = st.rc;
    const long long nc = 1ll << rc;
    const std::string ga = gather_expr(A), gb = gather_expr(B);
    const uint32_t nkk = 1u << st.nk;
    const int cexp = A.cexp + B.cexp;
    int lc = 0;
    while ((1 << lc) < cstep) ++lc;
    // block bits S among the high bits [lc, rc), the loop runs over the rest R
    std::vector<int> S, R;
    if (nc > (long long)cstep) {
        const uint32_t am = source_mask(A), bm = source_mask(B);
        std::vector<int> aonly, bonly, other;
        for (int bit = lc; bit < rc; ++bit) {
            const bool ia = (am >> bit) & 1u, ib = (bm >> bit) & 1u;
            if (ia && !ib) aonly.push_back(bit);
            else if (ib && !ia) bonly.push_back(bit);
            else other.push_back(bit);
        }
        int want = 0;
        while ((2 << want) <= std::max(1, block)) ++want;
        size_t ia = 0, ib = 0, io = 0;
        while ((int)S.size() < want && (ia < aonly.size() || ib < bonly.size() || io < other.size())) {
            if (ia < aonly.size() && (ia <= ib || ib >= bonly.size())) S.push_back(aonly[ia++]);
            else if (ib < bonly.size()) S.push_back(bonly[ib++]);
            else S.push_back(other[io++]);
        }
        for (int bit = lc; bit < rc; ++bit)
            if (std::find(S.begin(), S.end(), bit) == S.end()) R.push_back(bit);
    }
    const uint32_t am = source_mask(A), bm = source_mask(B);
    const int ns = (int)S.size();
    // subsets of S that matter to A / to B
    std::vector<uint32_t> acombo, bcombo;   // bit patterns (in output-index bits)
    auto subsets = [&](uint32_t mask) {
        std::vector<uint32_t> v;
        std::vector<int> bits;
        for (int x : S)
            if ((mask >> x) & 1u) bits.push_back(x);
        for (uint32_t t = 0; t < (1u << bits.size()); ++t) {
            uint32_t m = 0;
            for (size_t j = 0; j < bits.size(); ++j)
                if ((t >> j) & 1u) m |= 1u << bits[j];
            v.push_back(m);
        }
        return v;
    };
    acombo = subsets(am);
    bcombo = subsets(bm);
    std::ostringstream b;
    for (size_t x = 0; x < acombo.size(); ++x)
        b << "      const unsigned ar" << x << " = " << subst_c(ga, "c | " + std::to_string(acombo[x]) + "u") << ";\n";
    for (size_t y = 0; y < bcombo.size(); ++y)
        b << "      const unsigned br" << y << " = " << subst_c(gb, "c | " + std::to_string(bcombo[y]) + "u") << ";\n";
    // contraction terms in chunks of kch (all of them at once when short);
    // operand values loaded once per (row, k) of the chunk
    const uint32_t kch = std::min(nkk, kMaxUnrollK);
    const bool kloop = kch < nkk;
    const std::string ia = kloop ? "(ar%1 | (kb << " + std::to_string(A.kshift) + "))" : "ar%1";
    const std::string ib = kloop ? "(br%1 | (kb << " + std::to_string(B.kshift) + "))" : "br%1";
    auto idx_of = [](const std::string &pat, size_t v) {
        std::string s = pat;
        const size_t at = s.find("%1");
        return s.replace(at, 2, std::to_string(v));
    };
    std::vector<size_t> out_x, out_y;
    for (uint32_t t = 0; t < (1u << ns); ++t) {
        uint32_t m = 0;
        for (int j = 0; j < ns; ++j)
            if ((t >> j) & 1u) m |= 1u << S[j];
        out_x.push_back(std::find(acombo.begin(), acombo.end(), m & am) - acombo.begin());
        out_y.push_back(std::find(bcombo.begin(), bcombo.end(), m & bm) - bcombo.begin());
        b << "      T acc" << t << " = 0;\n";
    }
    if (kloop) b << "      #pragma unroll 1\n      for (unsigned kb = 0; kb < " << nkk << "u; kb += " << kch << "u) {\n";
    for (uint32_t k = 0; k < kch; ++k) {
        for (size_t x = 0; x < acombo.size(); ++x) {
            std::ostringstream pre;
            const std::string nm = idx_of(ia, x);
            const std::string tmp = "sa" + std::to_string(k) + "_" + std::to_string(x);
            const std::string v = load_expr(A, "pa", nm.c_str(), k << A.kshift, pre, tmp);
            b << pre.str();
            if (v != tmp) b << "      const T " << tmp << " = " << v << ";\n";
        }
        for (size_t y = 0; y < bcombo.size(); ++y) {
            std::ostringstream pre;
            const std::string nm = idx_of(ib, y);
            const std::string tmp = "sb" + std::to_string(k) + "_" + std::to_string(y);
            const std::string v = load_expr(B, "pb", nm.c_str(), k << B.kshift, pre, tmp);
            b << pre.str();
            if (v != tmp) b << "      const T " << tmp << " = " << v << ";\n";
        }
    }
    for (uint32_t t = 0; t < (1u << ns); ++t)
        for (uint32_t k = 0; k < kch; ++k)
            b << "      acc" << t << " = " << (fp64 ? "fma(" : "fmaf(") << "sa" << k << "_" << out_x[t] << ", sb" << k << "_"
              << out_y[t] << ", acc" << t << ");\n";
    if (kloop) b << "      }\n";
    // outputs of the block
    for (uint32_t t = 0; t < (1u << ns); ++t) {
        uint32_t m = 0;
        for (int j = 0; j < ns; ++j)
            if ((t >> j) & 1u) m |= 1u << S[j];
        const std::string acc = "acc" + std::to_string(t);
        if (fp64) {
            if (cexp != 0) b << "      " << acc << " = ldexp(" << acc << ", " << cexp << ");\n";
        } else {
            b << "      " << acc << " = ldexpf(" << acc << ", shift);\n";
            b << "      lmax = " << acc << " > lmax ? " << acc << " : lmax;\n";
        }
        b << "      pc[(c | " << m << "u) << GLOG] = " << acc << ";\n";
    }
    if (nc <= (long long)cstep) {
        o << "    if (c0 < " << nc << ") {\n      const unsigned c = (unsigned)c0;\n" << b.str() << "    }\n";
        return;
    }
    // c = c0 | deposit(i, R)
    std::string dep = "(unsigned)c0";
    for (size_t j = 0; j < R.size(); ++j)
        dep += " | (((i >> " + std::to_string(j) + ") & 1u) << " + std::to_string(R[j]) + ")";
    o << "    #pragma unroll 1\n";
    o << "    for (unsigned i = 0; i < " << (1u << R.size()) << "u; ++i) {\n";
    o << "      const unsigned c = " << dep << ";\n";
    o << b.str();
    o << "    }\n";
}

void emit_outputs_split_k(std::ostringstream &o, const StepDesc &st, int threads, int rb);

// Bits of `mask` (ascending).
std::vector<int> bits_of(uint32_t mask) {
    std::vector<int> v;
    for (int b = 0; b < 32; ++b)
        if ((mask >> b) & 1u) v.push_back(b);
    return v;
}

// `(x)` spread onto the given bit positions: bit t of x goes to pos[t].
std::string deposit(const std::string &x, const std::vector<int> &pos) {
    if (pos.empty()) return "0u";
    std::string r;
    for (size_t t = 0; t < pos.size(); ++t) {
        if (t) r += " | ";
        r += "(((" + x + ") >> " + std::to_string(t) + ") & 1u) << " + std::to_string(pos[t]);
    }
    return "(" + r + ")";
}

// The outputs of a step as described at split_k_block.  Thread t of the
// workgroup belongs to block t / thr and takes the terms k = t % thr, + thr, ..
// (thr = threads per block, so the k range of every thread ends inside 2^nk);
// the block's bits are the step's exclusive output bits first, so that an A
// value serves all B values of its k and the other way round.
void emit_outputs_split_k(std::ostringstream &o, const StepDesc &st, int threads, int rb) {
    const OperandDesc &A = st.a, &B = st.b;
    const uint32_t am = source_mask(A), bm = source_mask(B);
    const int rc = st.rc, thr = threads >> (rc - rb), waves = std::max(1, thr / 64);
    std::vector<int> aonly, bonly, other, S;
    for (int b = 0; b < rc; ++b) {
        const bool ia = (am >> b) & 1u, ib = (bm >> b) & 1u;
        (ia && !ib ? aonly : ib && !ia ? bonly : other).push_back(b);
    }
    size_t ia = 0, ib = 0, io = 0;
    while ((int)S.size() < rb) {
        if (ia < aonly.size() && (ia <= ib || ib >= bonly.size())) S.push_back(aonly[ia++]);
        else if (ib < bonly.size()) S.push_back(bonly[ib++]);
        else S.push_back(other[io++]);
    }
    std::vector<int> R;
    uint32_t sm = 0;
    for (int b : S) sm |= 1u << b;
    for (int b = 0; b < rc; ++b)
        if (!((sm >> b) & 1u)) R.push_back(b);
    auto combos = [&](uint32_t mask) {
        std::vector<int> bits;
        for (int b : S)
            if ((mask >> b) & 1u) bits.push_back(b);
        std::vector<uint32_t> v;
        for (uint32_t t = 0; t < (1u << bits.size()); ++t) v.push_back(pdep(t, bits));
        return v;
    };
    const std::vector<uint32_t> ca = combos(am), cb = combos(bm);
    auto single = [](const OperandDesc &op) { return op.kind == kInter ? 1u << op.nsingle : 1u; };
    const std::string ga = gather_expr(A), gb = gather_expr(B);
    o << "    {\n      float *red = reinterpret_cast<float *>(smem + RED);\n";
    o << "      const unsigned blk = (unsigned)tid / " << thr << "u, kl = (unsigned)tid % " << thr << "u;\n";
    o << "      const unsigned rb = " << (R.empty() ? std::string("0u") : deposit("blk", R)) << ";\n";
    for (size_t x = 0; x < ca.size(); ++x)
        o << "      const unsigned ar" << x << " = " << subst_c(ga, "(rb | " + std::to_string(ca[x]) + "u)") << ";\n";
    for (size_t y = 0; y < cb.size(); ++y)
        o << "      const unsigned br" << y << " = " << subst_c(gb, "(rb | " + std::to_string(cb[y]) + "u)") << ";\n";
    for (uint32_t t = 0; t < (1u << rb); ++t) o << "      float acc" << t << " = 0.f;\n";
    // two terms per iteration in flight (each thread has at least eight)
    o << "      #pragma unroll 2\n      for (unsigned k = kl; k < " << (1u << st.nk) << "u; k += " << thr << "u) {\n";
    auto loads = [&](const OperandDesc &op, const char *base, const char *r, const char *v, size_t n) {
        for (size_t x = 0; x < n; ++x) {
            const std::string idx = std::string(r) + std::to_string(x) + " | (k << " + std::to_string(op.kshift) + ")";
            o << "        float " << v << x << " = " << base << "[" << idx << "];\n";
            for (uint32_t q = 1; q < single(op); ++q)
                o << "        " << v << x << " += " << base << "[" << idx << " | " << (q << op.sshift) << "u];\n";
        }
    };
    loads(A, "pa", "ar", "va", ca.size());
    loads(B, "pb", "br", "vb", cb.size());
    std::vector<uint32_t> outs;
    for (uint32_t t = 0; t < (1u << rb); ++t) {
        const uint32_t c = pdep(t, S);
        outs.push_back(c);
        const size_t x = std::find(ca.begin(), ca.end(), c & am) - ca.begin();
        const size_t y = std::find(cb.begin(), cb.end(), c & bm) - cb.begin();
        o << "        acc" << t << " = fmaf(va" << x << ", vb" << y << ", acc" << t << ");\n";
    }
    o << "      }\n";
    for (uint32_t t = 0; t < (1u << rb); ++t) {
        for (int w = 1; w < std::min(thr, 64); w <<= 1) o << "      acc" << t << " += __shfl_xor(acc" << t << ", " << w << ");\n";
        o << "      if ((kl & 63u) == 0u) red[((kl >> 6) << " << rc << ") | rb | " << outs[t] << "u] = acc" << t << ";\n";
    }
    o << "      __syncthreads();\n";
    o << "      if (tid < " << (1 << rc) << ") {\n        float x = red[tid];\n";
    for (int w = 1; w < waves; ++w) o << "        x += red[" << (w << rc) << " + tid];\n";
    o << "        x = ldexpf(x, shift);\n        lmax = x > lmax ? x : lmax;\n        pc[tid] = x;\n      }\n    }\n";
}

// GEMM-shaped step on BF16 MFMA: per syndrome, C[i, j] = sum_k A[i, k] B[k, j]
// with i over the output bits that feed only A, j over those that feed only
// B, and the remaining output bits (shared, or beyond the 32 x 32 tile)
// enumerating tiles.  Operands are rounded to BF16 (nearest even) as they are
// read, the products accumulate in FP32 inside the MFMA, the output is scaled
// like every FP32 step.  Layouts (v_mfma_f32_32x32x16_bf16, wave64): lane l
// holds A[l % 32][8 (l / 32) .. +7], B[8 (l / 32) .. +7][l % 32], and
// D[8 (v / 4) + 4 (l / 32) + v % 4][l % 32] for v = 0..15.
void emit_outputs_mfma(std::ostringstream &o, const StepDesc &st, int threads) {
    const OperandDesc &A = st.a, &B = st.b;
    const uint32_t am = source_mask(A), bm = source_mask(B);
    const uint32_t outm = (st.rc >= 32) ? 0xffffffffu : ((1u << st.rc) - 1u);
    const std::vector<int> aon = bits_of(am & ~bm & outm), bon = bits_of(bm & ~am & outm);
    const std::vector<int> ai(aon.begin(), aon.begin() + 5), bj(bon.begin(), bon.begin() + 5);
    std::vector<int> rest;
    for (int b = 0; b < st.rc; ++b)
        if (std::find(ai.begin(), ai.end(), b) == ai.end() && std::find(bj.begin(), bj.end(), b) == bj.end())
            rest.push_back(b);
    const unsigned ntiles = 1u << rest.size();
    const int nwaves = threads / 64;
    const int chunks = 1 << (st.nk - 4);
    const std::string ga = gather_expr(A), gb = gather_expr(B);
    auto ld = [&](const OperandDesc &op, const char *base, const char *idx, const std::string &k) {
        const std::string e = std::string(idx) + " | ((" + k + ") << " + std::to_string(op.kshift) + ")";
        if (op.kind == kInter) return std::string(base) + "[(" + e + ") << GLOG]";
        return std::string(base) + "[" + e + "]";
    };
    o << "    {\n";
    o << "      const int l = tid & 63, w = tid >> 6;\n";
    o << "      for (unsigned t = (unsigned)w; t < " << ntiles << "u; t += " << nwaves << "u) {\n";
    o << "        const unsigned tb = " << deposit("t", rest) << ";\n";
    o << "        const unsigned ci = tb | " << deposit("(unsigned)(l & 31)", ai) << ";\n";
    o << "        const unsigned cj = tb | " << deposit("(unsigned)(l & 31)", bj) << ";\n";
    o << "        const unsigned ar = " << subst_c(ga, "ci") << ";\n";
    o << "        const unsigned br = " << subst_c(gb, "cj") << ";\n";
    o << "        f32x16 acc = {};\n";
    for (int ch = 0; ch < chunks; ++ch) {
        o << "        {\n          const unsigned kb = " << ch * 16 << "u + 8u * (unsigned)(l >> 5);\n";
        o << "          bf16x8 av, bv;\n";
        for (int e = 0; e < 8; ++e) {
            const std::string k = "kb + " + std::to_string(e) + "u";
            o << "          av[" << e << "] = (short)to_bf16(" << ld(A, "pa", "ar", k) << ");\n";
            o << "          bv[" << e << "] = (short)to_bf16(" << ld(B, "pb", "br", k) << ");\n";
        }
        o << "          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc, 0, 0, 0);\n        }\n";
    }
    o << "        #pragma unroll\n";
    o << "        for (int v = 0; v < 16; ++v) {\n";
    o << "          const unsigned i = 8u * (unsigned)(v >> 2) + 4u * (unsigned)(l >> 5) + (unsigned)(v & 3);\n";
    o << "          const unsigned c = tb | " << deposit("i", ai) << " | " << deposit("(unsigned)(l & 31)", bj) << ";\n";
    o << "          const float x = ldexpf(acc[v], shift);\n";
    o << "          lmax = x > lmax ? x : lmax;\n";
    o << "          pc[c << GLOG] = x;\n";
    o << "        }\n      }\n    }\n";
}

// Operand bit that output bit u feeds, or -1.
int seg_image(const OperandDesc &op, int u) {
    for (int i = 0; i < op.nseg; ++i) {
        const Seg &g = op.seg[i];
        if (g.width > 0 && u >= g.src && u < g.src + g.width) return g.dst + (u - g.src);
    }
    return -1;
}

// Exclusive output bits of a step: those feeding only A and only B.
void mfma_side_bits(const StepDesc &st, std::vector<int> &aon, std::vector<int> &bon) {
    const uint32_t am = source_mask(st.a), bm = source_mask(st.b);
    const uint32_t outm = (st.rc >= 32) ? 0xffffffffu : ((1u << st.rc) - 1u);
    aon = bits_of(am & ~bm & outm);
    bon = bits_of(bm & ~am & outm);
}

// GEMM-shaped step on FP32 MFMA, full FP32 operands: per syndrome
// C[i, j] = sum_k A[i, k] B[k, j] as above, in tiles of 32 x 32
// (v_mfma_f32_32x32x2f32, K = 2 per instruction) when both sides have five
// exclusive output bits, else 16 x 16 (v_mfma_f32_16x16x4f32, K = 4).  Each
// wave owns a block of ra x rb tiles (up to two more A-only output bits and
// one more B-only bit: 4 x 2 tiles, the best of 2 x 2, 4 x 2 and 2 x 4 on
// toric L=5; 4 x 4 spills), so every operand value a lane loads feeds rb (or
// ra) MFMAs.  The k loop takes ku instructions' worth of contracted values
// per iteration; a group's registers are loaded again for the next iteration as
// soon as its MFMAs have been issued, and the last iteration of a block loads
// the first values of the wave's next block, so that loads stay in flight
// across the block's stores (at one or two waves per SIMD few other waves hide
// them, and a wait for loads behind stores is a wait for the stores too).  The
// wave's last block loads its own first values once more, unused.  Measured
// against one wait per iteration for all of its loads: the circuit-level d=3,
// 3-round plan 357 -> 330 us per 16,384, d=5 with 2 rounds 2.91 -> 2.80 ms per
// 4,096, toric L=5 20.0 -> 19.7 ms per 512 (its widest step runs at 50 of 64
// multiply-adds per cycle and workgroup, the FP32 MFMA rate).
// Layouts (wave64), with T the tile edge (64 / T contracted values per
// instruction):
// lane l holds A[l % T][l / T] and B[l / T][l % T]; T = 32: D[v] =
// C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32], v = 0..15; T = 16: D[v] =
// C[4 (l / 16) + v][l % 16], v = 0..3.  Every index stays inside the
// operand and output ranges by construction (i, j < T over that many
// output bits, k < 2^nk, and every lane runs the same number of k
// iterations), so a layout mistake shows as wrong values, never as an
// out-of-range access.
void emit_outputs_mfma32(std::ostringstream &o, const StepDesc &st, int threads) {
    std::vector<int> aon, bon;
    mfma_side_bits(st, aon, bon);
    const bool big = aon.size() >= 5 && bon.size() >= 5;
    const int tbits = big ? 5 : 4;                 // tile edge 2^tbits
    // a store's lanes differ in the columns' bits: where the rows hold at least
    // three more of the output's low five (a cache line) the operands change
    // places, so that a store fills lines instead of touching up to 32 with a
    // float each (toric L=4, 2,048 syndromes: 13.8 -> 9.7 ms; 11.2 with such
    // stores but the operands loaded only after them)
    int low = 0;
    for (int t = 0; t < tbits; ++t) low += (aon[t] < 5) - (bon[t] < 5);
    const bool swap = low >= 3;
    if (swap) std::swap(aon, bon);
    const OperandDesc &A = swap ? st.b : st.a, &B = swap ? st.a : st.b;
    const std::string pa = swap ? "pb" : "pa", pb = swap ? "pa" : "pb";
    const unsigned tedge = 1u << tbits, kq = 64u / tedge;   // k values per instruction
    const std::vector<int> ai(aon.begin(), aon.begin() + tbits), bj(bon.begin(), bon.begin() + tbits);
    // a block shrinks while there are fewer blocks than waves: at 4 x 2 tiles a
    // 128 x 64 step is one block, and three of four waves would idle
    const int nwaves = threads / 64;
    int xa = std::min<int>(2, (int)aon.size() - tbits), xb = std::min<int>(1, (int)bon.size() - tbits);
    while (xa + xb > 0 && (1 << (st.rc - 2 * tbits - xa - xb)) < nwaves) (xa >= 2 * xb ? xa : xb) -= 1;
    const std::vector<int> a2(aon.begin() + tbits, aon.begin() + tbits + xa);
    const std::vector<int> b2(bon.begin() + tbits, bon.begin() + tbits + xb);
    std::vector<int> rest;
    for (int b = 0; b < st.rc; ++b) {
        const bool used = std::find(ai.begin(), ai.end(), b) != ai.end() ||
                          std::find(bj.begin(), bj.end(), b) != bj.end() ||
                          std::find(a2.begin(), a2.end(), b) != a2.end() ||
                          std::find(b2.begin(), b2.end(), b) != b2.end();
        if (!used) rest.push_back(b);
    }
    const int ra = 1 << xa, rb = 1 << xb;
    const unsigned ntiles = 1u << rest.size();
    const unsigned nkk = 1u << st.nk;
    const unsigned ku = std::min(4u, nkk / kq);   // instructions' k groups per loop iteration
    const unsigned kstep = kq * ku;
    const std::string tm = std::to_string(tedge - 1) + "u", lsh = std::to_string(tbits);
    const char *acc_t = big ? "f32x16" : "f32x4";
    const char *mfma = big ? "__builtin_amdgcn_mfma_f32_32x32x2f32" : "__builtin_amdgcn_mfma_f32_16x16x4f32";
    // Operand bits that output bits feed (those that feed the other side only
    // drop out), and the operand index made from them.
    auto image = [](const OperandDesc &op, const std::vector<int> &bits) {
        std::vector<int> v;
        for (int c : bits) v.push_back(seg_image(op, c));
        return v;
    };
    auto spread = [](const std::string &x, const std::vector<int> &pos) {
        std::string r;
        for (size_t t = 0; t < pos.size(); ++t)
            if (pos[t] >= 0)
                r += std::string(r.empty() ? "" : " | ") + "(((" + x + ") >> " + std::to_string(t) + ") & 1u) << " +
                     std::to_string(pos[t]);
        return r.empty() ? std::string("0u") : "(" + r + ")";
    };
    // place of a block's first operand values (the lane's row or column and its
    // contracted value within a group); the values of the block's other tiles
    // and groups lie at constant distances
    const std::string lane = "(unsigned)(l & " + tm + ")", kl = "((unsigned)(l >> " + lsh + ") << ";
    auto offsets = [&](const std::string &t) {
        return "          tb = " + deposit(t, rest) + ";\n          qa = " + pa + " + (" + spread(t, image(A, rest)) + " | " +
               spread(lane, image(A, ai)) + " | " + kl + std::to_string(A.kshift) + "));\n          qb = " + pb + " + (" +
               spread(t, image(B, rest)) + " | " + spread(lane, image(B, bj)) + " | " + kl + std::to_string(B.kshift) +
               "));\n";
    };
    auto load = [&](unsigned u) {
        for (int x = 0; x < ra; ++x)
            o << "          a" << u << "_" << x << " = qa[" << (pdep(x, image(A, a2)) + ((kq * u) << A.kshift)) << "];\n";
        for (int y = 0; y < rb; ++y)
            o << "          b" << u << "_" << y << " = qb[" << (pdep(y, image(B, b2)) + ((kq * u) << B.kshift)) << "];\n";
        // in this order, group by group: a wait for the oldest group is then not
        // a wait for all
        o << "          __builtin_amdgcn_sched_barrier(0);\n";
    };
    o << "    {\n";
    o << "      const int l = tid & 63, w = tid >> 6;\n";
    o << "      if (w < " << ntiles << ") {\n";
    o << "      unsigned tb;\n      const T *qa, *qb;\n      float a0_0";
    for (unsigned u = 0; u < ku; ++u) {
        for (int x = 0; x < ra; ++x)
            if (u || x) o << ", a" << u << "_" << x;
        for (int y = 0; y < rb; ++y) o << ", b" << u << "_" << y;
    }
    o << ";\n          " << offsets("(unsigned)w");
    for (unsigned u = 0; u < ku; ++u) load(u);
    o << "      #pragma unroll 1\n";
    o << "      for (unsigned t = (unsigned)w; t < " << ntiles << "u; t += " << nwaves << "u) {\n";
    o << "        const unsigned tc = tb;\n";
    for (int x = 0; x < ra; ++x)
        for (int y = 0; y < rb; ++y) o << "        " << acc_t << " acc" << x << "_" << y << " = {};\n";
    o << "        #pragma unroll 1\n";
    o << "        for (unsigned kb = " << kstep << "u; kb <= " << nkk << "u; kb += " << kstep << "u) {\n";
    o << "          if (kb < " << nkk << "u) {\n";
    o << "            qa += " << (kstep << A.kshift) << ";\n            qb += " << (kstep << B.kshift) << ";\n";
    o << "          } else {\n          const unsigned tn = t + " << nwaves << "u < " << ntiles << "u ? t + " << nwaves
      << "u : t;\n          " << offsets("tn") << "          }\n";
    for (unsigned u = 0; u < ku; ++u) {
        for (int x = 0; x < ra; ++x)
            for (int y = 0; y < rb; ++y)
                o << "          acc" << x << "_" << y << " = " << mfma << "(a" << u << "_" << x << ", b" << u << "_" << y
                  << ", acc" << x << "_" << y << ", 0, 0, 0);\n";
        load(u);
    }
    o << "        }\n";
    for (int x = 0; x < ra; ++x)
        for (int y = 0; y < rb; ++y) {
            o << "        #pragma unroll\n";
            o << "        for (int v = 0; v < " << (big ? 16 : 4) << "; ++v) {\n";
            if (big)
                o << "          const unsigned i = 8u * (unsigned)(v >> 2) + 4u * (unsigned)(l >> 5) + (unsigned)(v & 3);\n";
            else
                o << "          const unsigned i = 4u * (unsigned)(l >> 4) + (unsigned)v;\n";
            o << "          const unsigned c = tc | " << deposit("i", ai) << " | " << deposit(std::to_string(x) + "u", a2)
              << " | " << deposit("(unsigned)(l & " + tm + ")", bj) << " | " << deposit(std::to_string(y) + "u", b2)
              << ";\n";
            o << "          const float x = ldexpf(acc" << x << "_" << y << "[v], shift);\n";
            o << "          lmax = x > lmax ? x : lmax;\n";
            o << "          pc[c << GLOG] = x;\n";
            o << "        }\n";
        }
    o << "      }\n      }\n    }\n";
}

void emit_step(std::ostringstream &o, const StepDesc &st, int s, size_t const_n, int cstep, bool fp64, int unroll,
               const SpecCfg *mfma_cfg, const Places &places, bool opaque_tid = false) {
    const OperandDesc &A = st.a, &B = st.b;
    int64_t lds[2] = {-1, -1};
    for (int side = 0; side < 2; ++side)
        if (places.prod[s][side] >= 0) lds[side] = places.lds[places.prod[s][side]];
    const int64_t lc = places.lds[s];
    const std::string pc = (lc >= 0 ? "lwork + " + std::to_string(lc) : "work + " + std::to_string((long long)st.c_off)) +
                           " * G + g;\n";
    o << "  { // step " << s << ": rank " << st.rc << ", contracted " << st.nk << "\n";
    if (opaque_tid)
        // the step's own copy of the thread index, opaque to the optimiser:
        // nothing derived from it is hoisted out of the kernel's loop over
        // tiles or shared with other steps, so per-thread index values live
        // for one step only
        o << "    int tid = (int)threadIdx.x;\n    asm volatile(\"\" : \"+v\"(tid));\n"
             "    const int g = tid & (G - 1), c0 = tid >> GLOG, lane = tid & 63;\n"
             "    (void)g; (void)c0; (void)lane;\n";
    if (fp64) {
        // generic FP64 step: no scaling, the folded constant exponents restored per entry
        emit_base(o, "pa", A, const_n, lds[0]);
        emit_base(o, "pb", B, const_n, lds[1]);
        o << "    T *pc = " << pc;
        emit_outputs(o, st, cstep, unroll, true);
        o << "  }\n";
        o << "  __syncthreads();\n";
        return;
    }
    o << "    int ea, eb, na = 0, nb = 0;\n";
    for (int side = 0; side < 2; ++side) {
        const OperandDesc &op = side ? B : A;
        const char *n = side ? "nb" : "na";
        const char *e = side ? "eb" : "ea";
        if (op.kind == kInter) {
            o << "    { const float m = __uint_as_float((unsigned)(mx[" << op.slot
              << " * G + g] & 0xffffffffull)); " << n << " = (m > 0.f) ? ilogbf(m) : 0; " << e << " = ex["
              << op.slot << " * G + g] + " << n << "; }\n";
        } else {
            o << "    " << e << " = " << op.cexp << ";\n";
        }
    }
    o << "    const int shift = -(na + nb);\n";
    {
        std::string cond;
        if (A.kind == kInter) cond += "na < -100";
        if (B.kind == kInter) cond += std::string(cond.empty() ? "" : " || ") + "nb < -100";
        if (!cond.empty()) o << "    if (" << cond << ") lowf[g] = 1;\n";
    }
    emit_base(o, "pa", A, const_n, lds[0]);
    emit_base(o, "pb", B, const_n, lds[1]);
    o << "    T *pc = " << pc;
    o << "    T lmax = 0;\n";
    // a slab's steps of one or two contracted labels wait on memory: more
    // outputs per lane block put more loads in flight (circuit-level d=5, 2
    // rounds 3.18 -> 2.91 ms per 4,096 against blocks of 4)
    if (opaque_tid && st.nk <= 2) unroll = std::max(unroll, st.nk <= 1 ? 16 : 8);
    if (mfma_cfg && spec_step_uses_mfma(st, *mfma_cfg))
        emit_outputs_mfma(o, st, mfma_cfg->threads);
    else if (mfma_cfg && spec_step_uses_mfma32(st, *mfma_cfg))
        emit_outputs_mfma32(o, st, mfma_cfg->threads);
    else if (mfma_cfg && split_k_block(st, *mfma_cfg) >= 0)
        emit_outputs_split_k(o, st, mfma_cfg->threads, split_k_block(st, *mfma_cfg));
    else
        emit_outputs(o, st, cstep, unroll, false);
    o << "    for (int w = G; w < 64; w <<= 1) { const float other = __shfl_xor(lmax, w); lmax = other > lmax ? other : lmax; }\n";
    o << "    if (lane < G) atomicMax(&mx[" << st.c_slot << " * G + g], ((unsigned long long)(tag_base + " << s
      << "u) << 32) | (unsigned long long)__float_as_uint(lmax));\n";
    o << "    if (tid < G) ex[" << st.c_slot << " * G + g] = ea + eb;\n";
    o << "  }\n";
    o << "  __syncthreads();\n";
}

// ---- register-resident variant ------------------------------------------
//
// A quad of lanes owns one syndrome.  Tensor X of rank r keeps entry i in
// lane sum_t bit(i, pos[t]) << t of the quad and in register pext(i, other
// bits) of that lane; a missing pos[t] replicates X along lane bit t.  The
// consumer of X chooses X's lane bits: an output lane bit that feeds X is
// placed in the same lane slot of X, so those index bits never cross lanes
// and the register an operand entry lives in never depends on the lane.  A
// fetch is then one DPP quad permutation (or a plain register read when the
// permutation is the identity).  Layouts are decided from the root down.

struct RLay {
    int pos[2] = {-1, -1};   // tensor index bit held by lane bit t (-1: replicated along t)
};

uint32_t gather_host(uint32_t c, const OperandDesc &op) {
    uint32_t r = 0;
    for (int i = 0; i < op.nseg; ++i) {
        const Seg &g = op.seg[i];
        if (g.width <= 0) continue;
        const uint32_t w = (g.width >= 32) ? 0xffffffffu : ((1u << g.width) - 1u);
        r |= ((c >> g.src) & w) << g.dst;
    }
    return r;
}

int lane_bits(const RLay &l) { return (l.pos[0] >= 0) + (l.pos[1] >= 0); }

std::vector<int> reg_bits(const RLay &l, int rank) {
    std::vector<int> v;
    for (int b = 0; b < rank; ++b)
        if (b != l.pos[0] && b != l.pos[1]) v.push_back(b);
    return v;
}

uint32_t pext(uint32_t x, const std::vector<int> &bits) {
    uint32_t r = 0;
    for (size_t j = 0; j < bits.size(); ++j) r |= ((x >> bits[j]) & 1u) << j;
    return r;
}

// Registers per lane above which the variant is not offered (512 VGPRs and
// AGPRs per lane at one wave per SIMD, less the step temporaries).
constexpr int kRegBudget = 400;

struct RegPlan {
    std::vector<int> prod[2];   // producing step of each step's intermediate A / B, or -1
    std::vector<RLay> lay;      // per step output
    int root = -1;
    int peak = 0;               // live tensor registers per lane
    std::string err;
};

// Live tensor registers per lane in execution order; false above the budget.
bool reg_peak_ok(const CompiledPlan &cp, RegPlan &rp) {
    int live = 0;
    rp.peak = 0;
    for (int s = 0; s < (int)cp.steps.size(); ++s) {
        const StepDesc &st = cp.steps[s];
        live += 1 << (st.rc - lane_bits(rp.lay[s]));
        rp.peak = std::max(rp.peak, live);
        for (int side = 0; side < 2; ++side) {
            const int p = rp.prod[side][s];
            if (p >= 0) live -= 1 << (cp.steps[p].rc - lane_bits(rp.lay[p]));
        }
    }
    if (rp.peak > kRegBudget) return rp.err = "more live tensor entries per lane than registers", false;
    return true;
}

// quad_perm control: destination lane d of each quad reads lane src[d]
int quad_ctrl(const int src[4]) { return src[0] | (src[1] << 2) | (src[2] << 4) | (src[3] << 6); }

constexpr int kIdentityCtrl = 0xE4;   // quad_perm [0, 1, 2, 3]

// DPP control with which a consumer writing layout LC reads entry `idx`
// (lane-independent bits) of operand `op` stored in layout LX; -1 when an
// output lane bit that feeds the operand does not sit in the same lane slot
// of LX (the register would then depend on the lane).
int fetch_ctrl(const OperandDesc &op, const RLay &LC, const RLay &LX, uint32_t idx) {
    int img[2];
    for (int t = 0; t < 2; ++t) {
        img[t] = LC.pos[t] >= 0 ? seg_image(op, LC.pos[t]) : -1;
        if (img[t] >= 0 && img[t] != LX.pos[t]) return -1;
    }
    int src[4];
    for (int d = 0; d < 4; ++d) {
        src[d] = 0;
        for (int t = 0; t < 2; ++t) {
            const int bit = (LX.pos[t] < 0 || img[t] >= 0) ? (d >> t) & 1 : (int)((idx >> LX.pos[t]) & 1u);
            src[d] |= bit << t;
        }
    }
    return quad_ctrl(src);
}

// Per-lane instruction estimate of one operand's reads in a step writing
// layout LC: distinct DPP moves (intermediate stored in *LX) or distinct
// table loads (LX null), summed over the contraction index as the emitter
// caches them.  -1 when LX is not a legal layout for this consumer.
long fetch_cost(const StepDesc &st, int side, const RLay &LC, const RLay *LX) {
    const OperandDesc &op = side ? st.b : st.a;
    if (LX)
        for (int t = 0; t < 2; ++t)
            if (LC.pos[t] >= 0) {
                const int img = seg_image(op, LC.pos[t]);
                if (img >= 0 && img != LX->pos[t]) return -1;
            }
    const std::vector<int> RB = reg_bits(LC, st.rc);
    const std::vector<int> RX = LX ? reg_bits(*LX, op.rank) : std::vector<int>();
    const uint32_t nreg = 1u << RB.size(), nkk = 1u << st.nk;
    const uint32_t nq = (LX && op.nsingle) ? (1u << op.nsingle) : 1u;
    long cost = 0;
    std::vector<uint64_t> keys;
    for (uint32_t k = 0; k < nkk; ++k) {
        keys.clear();
        for (uint32_t r = 0; r < nreg; ++r) {
            const uint32_t base = gather_host(pdep(r, RB), op) | (k << op.kshift);
            if (!LX) {
                keys.push_back(base);
                continue;
            }
            for (uint32_t q = 0; q < nq; ++q) {
                const uint32_t idx = base | (q << op.sshift);
                const int ctrl = fetch_ctrl(op, LC, *LX, idx);
                if (ctrl != kIdentityCtrl) keys.push_back(((uint64_t)pext(idx, RX) << 8) | (uint64_t)ctrl);
            }
        }
        std::sort(keys.begin(), keys.end());
        cost += (long)(std::unique(keys.begin(), keys.end()) - keys.begin());
    }
    return cost;
}

std::vector<RLay> layout_candidates(int rank) {
    std::vector<RLay> v;
    for (int a = -1; a < rank; ++a)
        for (int b = -1; b < rank; ++b) {
            if (a >= 0 && a == b) continue;
            RLay L;
            L.pos[0] = a;
            L.pos[1] = b;
            v.push_back(L);
        }
    return v;
}

// Lane layouts minimising the per-lane instruction estimate of the whole
// step program: for every step and output layout, its multiply-adds, scale
// and maximum per output register and table loads, plus for each
// intermediate operand the cheapest legal layout of it (its DPP moves here
// plus the best cost of its own subtree in that layout).  Exact over the
// tree (each tensor has one consumer); replication (a missing lane bit) is
// one of the options.  Only for tensors of rank <= 9.
bool reg_layout_dp(const CompiledPlan &cp, RegPlan &rp) {
    const int ns = (int)cp.steps.size();
    for (const StepDesc &st : cp.steps)
        if (st.rc > 9) return false;
    std::vector<std::vector<RLay>> cand(ns);
    std::vector<std::vector<long>> best(ns);
    std::vector<std::vector<std::array<int, 2>>> arg(ns);
    for (int s = 0; s < ns; ++s) {
        const StepDesc &st = cp.steps[s];
        cand[s] = layout_candidates(st.rc);
        best[s].assign(cand[s].size(), -1);
        arg[s].assign(cand[s].size(), {-1, -1});
        const long nkk = 1l << st.nk;
        for (size_t i = 0; i < cand[s].size(); ++i) {
            const RLay &L = cand[s][i];
            long total = (1l << (st.rc - lane_bits(L))) * (nkk + 2);
            bool ok = true;
            for (int side = 0; side < 2 && ok; ++side) {
                const int p = rp.prod[side][s];
                if (p < 0) {
                    total += fetch_cost(st, side, L, nullptr);
                    continue;
                }
                long bc = -1;
                int bj = -1;
                for (size_t j = 0; j < cand[p].size(); ++j) {
                    if (best[p][j] < 0) continue;
                    const long c = fetch_cost(st, side, L, &cand[p][j]);
                    if (c < 0) continue;
                    if (bc < 0 || c + best[p][j] < bc) {
                        bc = c + best[p][j];
                        bj = (int)j;
                    }
                }
                if (bj < 0) ok = false;
                total += bc;
                arg[s][i][side] = bj;
            }
            if (ok) best[s][i] = total;
        }
    }
    int bi = -1;
    for (size_t i = 0; i < cand[rp.root].size(); ++i)
        if (best[rp.root][i] >= 0 && (bi < 0 || best[rp.root][i] < best[rp.root][bi])) bi = (int)i;
    if (bi < 0) return false;
    std::vector<int> choice(ns, -1);
    choice[rp.root] = bi;
    for (int s = ns - 1; s >= 0; --s) {
        if (choice[s] < 0) return false;
        rp.lay[s] = cand[s][choice[s]];
        for (int side = 0; side < 2; ++side)
            if (rp.prod[side][s] >= 0) choice[rp.prod[side][s]] = arg[s][choice[s]][side];
    }
    return true;
}

bool reg_plan(const CompiledPlan &cp, RegPlan &rp) {
    const int ns = (int)cp.steps.size();
    if (ns == 0) return rp.err = "no per-syndrome steps", false;
    if (cp.n_out > 4) return rp.err = "more than 16 classes", false;
    rp.prod[0].assign(ns, -1);
    rp.prod[1].assign(ns, -1);
    rp.lay.assign(ns, RLay());
    std::vector<int> uses(ns, 0);
    for (int s = 0; s < ns; ++s) {
        const StepDesc &st = cp.steps[s];
        if (st.rc > 16) return rp.err = "tensor too wide for registers", false;
        for (int side = 0; side < 2; ++side) {
            const OperandDesc &op = side ? st.b : st.a;
            if (op.kind != kInter) continue;
            int p = -1;
            for (int j = s - 1; j >= 0; --j)
                if (cp.steps[j].c_off == op.off) {
                    p = j;
                    break;
                }
            if (p < 0 || cp.steps[p].rc != op.rank) return rp.err = "operand without a producing step", false;
            rp.prod[side][s] = p;
            ++uses[p];
        }
        if (st.is_root) rp.root = s;
    }
    if (rp.root < 0 || cp.steps[rp.root].c_off != cp.root_off || cp.steps[rp.root].rc != cp.n_out)
        return rp.err = "root step not found", false;
    for (int s = 0; s < ns; ++s)
        if (uses[s] != (s == rp.root ? 0 : 1)) return rp.err = "step output not used exactly once", false;
    if (cp.reg_checked && cp.reg_lay.empty()) return rp.err = cp.reg_err, false;
    if (cp.reg_lay.size() == 2 * (size_t)ns) {
        // prepared with the plan (spec_reg_prepare)
        for (int s = 0; s < ns; ++s) {
            rp.lay[s].pos[0] = cp.reg_lay[2 * s];
            rp.lay[s].pos[1] = cp.reg_lay[2 * s + 1];
        }
        return reg_peak_ok(cp, rp);
    }
    if (reg_layout_dp(cp, rp) && reg_peak_ok(cp, rp)) return true;
    rp.err.clear();
    rp.peak = 0;
    // greedy layouts, consumers first
    RLay &lr = rp.lay[rp.root];
    for (int t = 0; t < 2; ++t)
        if (cp.steps[rp.root].rc > t) lr.pos[t] = t;
    for (int s = ns - 1; s >= 0; --s) {
        const StepDesc &st = cp.steps[s];
        const RLay LC = rp.lay[s];
        for (int side = 0; side < 2; ++side) {
            const int p = rp.prod[side][s];
            if (p < 0) continue;
            const OperandDesc &op = side ? st.b : st.a;
            RLay L;
            for (int t = 0; t < 2; ++t)
                if (LC.pos[t] >= 0) L.pos[t] = seg_image(op, LC.pos[t]);
            // free slots: the bit that feeds most of the producer's intermediate operands
            const StepDesc &ps = cp.steps[p];
            for (int t = 0; t < 2; ++t) {
                if (L.pos[t] >= 0) continue;
                int best = -1, best_score = -1;
                for (int v = 0; v < op.rank; ++v) {
                    if (v == L.pos[0] || v == L.pos[1]) continue;
                    int score = 0;
                    if (ps.a.kind == kInter && seg_image(ps.a, v) >= 0) ++score;
                    if (ps.b.kind == kInter && seg_image(ps.b, v) >= 0) ++score;
                    if (score > best_score) {
                        best = v;
                        best_score = score;
                    }
                }
                L.pos[t] = best;
            }
            rp.lay[p] = L;
        }
    }
    return reg_peak_ok(cp, rp);
}

// Expression for entry `idx` (lane-independent bits) of intermediate X, made
// by step p with layout LX, read by a consumer with output layout LC.
bool reg_fetch(const OperandDesc &op, const RLay &LC, const RLay &LX, int p, uint32_t idx, std::string &out,
               std::string &err) {
    const int ctrl = fetch_ctrl(op, LC, LX, idx);
    if (ctrl < 0) return err = "lane bit of an operand moved", false;
    const std::string name = "x" + std::to_string(p) + "_" + std::to_string(pext(idx, reg_bits(LX, op.rank)));
    out = (ctrl == kIdentityCtrl) ? name : "QP(" + name + ", " + std::to_string(ctrl) + ")";
    return true;
}

// Plan-time scaling of the register-resident FP32 kernel (static mode).
//
// Every entry of every table is non-negative, so contracting the plan in
// FP64 with each sliced table replaced by the sum of its variants (the
// evidence of all syndromes at once) bounds every intermediate entry of every
// syndrome from above (ub).  The kernel stores intermediate X as
// X_true * 2^-E_X, E_X being the sum of the folded exponents of X's tables
// plus any static shifts below it.  A step shifts its output (one multiply
// per output register) only where its pre-shift bound
// log2 max ub - (E_a + E_b) would leave [kShiftLo, kShiftHi], so every value
// and every partial sum stays below 2^127 whatever the syndrome, and the
// plan is refused (the dynamic mode is used instead) when a bound cannot be
// kept below kOverflow.
//
// Underflow: an operation whose result drops below FP32's normal range errs
// by at most 2^-126 of its unit 2^E; carried to the root by the environment
// bound (env: the adjoint of the ub contraction, again over all syndromes),
// all of them together err by at most errsum in absolute terms (true
// units), also counting the FP32 rounding of the tables.  A syndrome whose
// largest root entry is below 2^theta, theta = log2 errsum + kErrBits, is
// re-checked in FP64, so accepted marginals err by at most 2^-kErrBits of
// the row maximum from underflow: one comparison at the root replaces the
// per-step maxima, exponents and rescales of the dynamic mode.
struct RegScale {
    std::vector<int> shift;   // per step: output scaled by 2^-shift
    std::vector<int> E;       // per step: exponent of the stored values
    std::vector<double> pre;  // per step: pre-shift bound, log2
    int e_root = 0;
    double theta = 0;         // log2 of the smallest root maximum accepted without re-check
};

constexpr double kShiftHi = 60, kShiftLo = -30, kOverflow = 120, kErrBits = 21;

// True values (in memory order) of a table operand, summed over its
// variants for a sliced one.
std::vector<double> table_bound(const CompiledPlan &cp, const OperandDesc &op) {
    const size_t n = size_t(1) << op.rank;
    std::vector<double> v(n, 0.0);
    const double sc = std::ldexp(1.0, op.cexp);
    if (op.kind == kConst) {
        for (size_t i = 0; i < n; ++i) v[i] = cp.const_pool[(size_t)op.off + i] * sc;
    } else {
        for (uint32_t var = 0; var < (1u << op.nev); ++var)
            for (size_t i = 0; i < n; ++i) v[i] += cp.sliced_pool[(size_t)op.off + ((size_t)var << op.rank) + i] * sc;
    }
    return v;
}

bool reg_static_scales(const CompiledPlan &cp, const RegPlan &rp, RegScale &rs, std::string &err) {
    const int ns = (int)cp.steps.size();
    std::vector<std::vector<double>> ub(ns), env(ns);
    std::vector<std::array<std::vector<double>, 2>> opv(ns);
    std::vector<std::array<int, 2>> opE(ns);
    rs.shift.assign(ns, 0);
    rs.E.assign(ns, 0);
    rs.pre.assign(ns, 0);
    auto lg = [](const std::vector<double> &v) {
        double m = 0;
        for (double x : v) m = std::max(m, x);
        return m > 0 ? std::log2(m) : -HUGE_VAL;
    };
    // forward: upper bounds and exponents
    for (int s = 0; s < ns; ++s) {
        const StepDesc &st = cp.steps[s];
        for (int side = 0; side < 2; ++side) {
            const OperandDesc &op = side ? st.b : st.a;
            const int p = rp.prod[side][s];
            opv[s][side] = p >= 0 ? ub[p] : table_bound(cp, op);
            opE[s][side] = p >= 0 ? rs.E[p] : op.cexp;
            const double single = lg(opv[s][side]) - opE[s][side] + op.nsingle;
            if (single > kOverflow) return err = "operand bound too large for static scaling", false;
        }
        const OperandDesc &A = st.a, &B = st.b;
        const std::vector<double> &va = opv[s][0], &vb = opv[s][1];
        std::vector<double> &c = ub[s];
        c.assign(size_t(1) << st.rc, 0.0);
        for (uint32_t ci = 0; ci < (1u << st.rc); ++ci) {
            const uint32_t ia = gather_host(ci, A), ib = gather_host(ci, B);
            double acc = 0;
            for (uint32_t k = 0; k < (1u << st.nk); ++k) {
                double sa = 0, sb = 0;
                for (uint32_t q = 0; q < (1u << A.nsingle); ++q) sa += va[ia | (q << A.sshift) | (k << A.kshift)];
                for (uint32_t q = 0; q < (1u << B.nsingle); ++q) sb += vb[ib | (q << B.sshift) | (k << B.kshift)];
                acc += sa * sb;
            }
            c[ci] = acc;
        }
        const int eab = opE[s][0] + opE[s][1];
        const double pre = lg(c) - eab;
        if (!(pre < HUGE_VAL)) return err = "non-finite bound", false;
        rs.pre[s] = pre;
        int sh = 0;
        if (pre > kShiftHi || (pre < kShiftLo && pre > -HUGE_VAL)) sh = (int)std::floor(pre);
        if (pre > kOverflow) return err = "step bound too large for static scaling", false;
        rs.shift[s] = sh;
        rs.E[s] = eab + sh;
    }
    // adjoint: environment bounds, and the underflow error they carry
    env[rp.root].assign(size_t(1) << cp.steps[rp.root].rc, 1.0);
    double errsum = 0;
    for (int s = ns - 1; s >= 0; --s) {
        const StepDesc &st = cp.steps[s];
        const OperandDesc &A = st.a, &B = st.b;
        const std::vector<double> &va = opv[s][0], &vb = opv[s][1], &ec = env[s];
        std::vector<double> ea(va.size(), 0.0), eb(vb.size(), 0.0);
        double envsum = 0;
        for (uint32_t ci = 0; ci < (1u << st.rc); ++ci) {
            envsum += ec[ci];
            const uint32_t ia = gather_host(ci, A), ib = gather_host(ci, B);
            for (uint32_t k = 0; k < (1u << st.nk); ++k) {
                double sa = 0, sb = 0;
                for (uint32_t q = 0; q < (1u << A.nsingle); ++q) sa += va[ia | (q << A.sshift) | (k << A.kshift)];
                for (uint32_t q = 0; q < (1u << B.nsingle); ++q) sb += vb[ib | (q << B.sshift) | (k << B.kshift)];
                for (uint32_t q = 0; q < (1u << A.nsingle); ++q) ea[ia | (q << A.sshift) | (k << A.kshift)] += ec[ci] * sb;
                for (uint32_t q = 0; q < (1u << B.nsingle); ++q) eb[ib | (q << B.sshift) | (k << B.kshift)] += ec[ci] * sa;
            }
        }
        // this step's operations: per output entry 2^nk products and the
        // single-side sums, each within 2^-126 of its unit when it underflows
        const double ops = std::ldexp(1.0, st.nk) * (1.0 + std::ldexp(1.0, A.nsingle) + std::ldexp(1.0, B.nsingle));
        const int unit = opE[s][0] + opE[s][1] + std::max(rs.shift[s], 0);
        errsum += ops * envsum * std::ldexp(1.0, unit - 126);
        for (int side = 0; side < 2; ++side) {
            const std::vector<double> &e = side ? eb : ea;
            const int p = rp.prod[side][s];
            if (p >= 0) {
                env[p] = e;
            } else {
                // FP32 rounding of the table's entries below the normal range
                double es = 0;
                for (double x : e) es += x;
                errsum += es * std::ldexp(1.0, opE[s][side] - 126);
            }
        }
    }
    if (!std::isfinite(errsum)) return err = "non-finite error bound", false;
    rs.e_root = rs.E[rp.root];
    rs.theta = errsum > 0 ? std::log2(errsum) + kErrBits : -HUGE_VAL;
    return true;
}

// The register-resident kernel is one straight line of code, cut into chunks:
// the terms of one contracted value of one step.  A chunk's table values are
// loaded several chunks before its multiply-adds (emit_reg_chunks).
constexpr int kPrefetch32 = 24, kPrefetch64 = 8;   // table values in flight

struct RegChunk {
    std::string loads;   // the step's table addresses (first chunk) and this chunk's table values
    int values = 0;      // table values loaded
    std::string body;
};

// One step of the register-resident kernel.  FP32 with `rs`: the static
// exponents and shifts of reg_static_scales; FP32 without: per-tensor
// power-of-two scaling from each operand's maximum (the generic FP32
// kernel's); FP64 (`fp64`): no scaling, the constant exponents folded out of
// table data restored per entry (the generic FP64 kernel's).
bool emit_reg_step(std::vector<RegChunk> &out, const CompiledPlan &cp, const RegPlan &rp, int s, size_t const_n,
                   bool fp64, const RegScale *rs, std::string &err) {
    const StepDesc &st = cp.steps[s];
    const RLay &LC = rp.lay[s];
    const std::vector<int> RB = reg_bits(LC, st.rc);
    const uint32_t nreg = 1u << RB.size();
    const uint32_t nkk = 1u << st.nk;
    const char *T = fp64 ? "double" : "float";
    const char *zero = fp64 ? "0.0" : "0.f";
    const bool dyn = !fp64 && !rs;
    const std::string S = std::to_string(s);
    const char *ab[2] = {"a", "b"};
    std::ostringstream first, addr;
    // the step program is a scope of its own, which the first step opens
    first << (s == 0 ? "    { // step " : "    // step ") << s << ": rank " << st.rc << ", contracted " << st.nk << ", " << nreg << " registers per lane";
    if (rs) first << "; bound 2^" << (int)std::ceil(rs->pre[s]) << " before a shift of " << rs->shift[s] << ", exponent "
                  << rs->E[s];
    first << "\n    " << T;
    for (uint32_t r = 0; r < nreg; ++r) first << (r ? ", " : " ") << "x" << s << "_" << r << " = " << zero;
    first << ";\n";
    for (int side = 0; side < 2 && dyn; ++side) {
        const OperandDesc &op = side ? st.b : st.a;
        const int p = rp.prod[side][s];
        if (op.kind == kInter)
            first << "    const int n" << ab[side] << S << " = (m" << p << " > 0.f) ? ilogbf(m" << p << ") : 0, e" << ab[side]
                  << S << " = e" << p << " + n" << ab[side] << S << ";\n";
        else
            first << "    const int n" << ab[side] << S << " = 0, e" << ab[side] << S << " = " << op.cexp << ";\n";
    }
    if (dyn) {
        first << "    const int shift" << S << " = -(na" << S << " + nb" << S << ");\n";
        std::string cond;
        if (st.a.kind == kInter) cond += "na" + S + " < -100";
        if (st.b.kind == kInter) cond += std::string(cond.empty() ? "" : " || ") + "nb" + S + " < -100";
        if (!cond.empty()) first << "    if (" << cond << ") lowf = 1;\n";
    }
    bool has_lane_off[2] = {false, false};
    for (int side = 0; side < 2; ++side) {
        const OperandDesc &op = side ? st.b : st.a;
        if (op.kind == kInter) continue;
        if (op.kind == kConst) {
            addr << "    const " << T << " *p" << ab[side] << S << " = tab + " << (long long)op.off << ";\n";
        } else {
            addr << "    const unsigned v" << ab[side] << S << " = 0u";
            for (int j = 0; j < op.nev; ++j) addr << " | (s" << op.ev_bit[j] << " << " << j << ")";
            addr << ";\n    const " << T << " *p" << ab[side] << S << " = tab + " << (long long)(const_n + (size_t)op.off)
                 << " + (v" << ab[side] << S << " << " << op.rank << ");\n";
        }
        std::string lo;
        for (int t = 0; t < 2; ++t) {
            if (LC.pos[t] < 0) continue;
            const uint32_t gbit = gather_host(1u << LC.pos[t], op);
            if (!gbit) continue;
            int sh = 0;
            while ((1u << sh) != gbit) ++sh;
            lo += std::string(lo.empty() ? "" : " | ") + "((((unsigned)q >> " + std::to_string(t) + ") & 1u) << " +
                  std::to_string(sh) + ")";
        }
        if (!lo.empty()) {
            addr << "    const unsigned l" << ab[side] << S << " = " << lo << ";\n";
            has_lane_off[side] = true;
        }
    }
    int ntmp = 0;
    for (uint32_t k = 0; k < nkk; ++k) {
        RegChunk chunk;
        std::ostringstream o, ld;
        if (k == 0) {
            o << first.str();
            ld << addr.str();
        }
        std::vector<std::pair<std::string, std::string>> cache;   // expression -> temporary
        auto temp = [&]() { return "f" + S + "_" + std::to_string(ntmp++); };
        auto value = [&](int side, uint32_t cst, std::string &name) -> bool {
            const OperandDesc &op = side ? st.b : st.a;
            const uint32_t idx = gather_host(cst, op) | (k << op.kshift);
            std::string expr;
            if (op.kind != kInter) {
                expr = std::string("p") + ab[side] + S + "[" +
                       (has_lane_off[side] ? std::string("l") + ab[side] + S + " + " : "") + std::to_string(idx) + "u]";
            } else {
                const int p = rp.prod[side][s];
                if (op.nsingle == 0) {
                    if (!reg_fetch(op, LC, rp.lay[p], p, idx, expr, err)) return false;
                    if (expr.compare(0, 3, "QP(") != 0) {
                        name = expr;
                        return true;
                    }
                } else {
                    // single-side labels summed first, ascending (as the generic kernel)
                    expr = "S";
                    std::vector<std::string> terms;
                    for (uint32_t qq = 0; qq < (1u << op.nsingle); ++qq) {
                        std::string t1;
                        if (!reg_fetch(op, LC, rp.lay[p], p, idx | (qq << op.sshift), t1, err)) return false;
                        terms.push_back(t1);
                        expr += "|" + t1;
                    }
                    for (auto &c : cache)
                        if (c.first == expr) {
                            name = c.second;
                            return true;
                        }
                    const std::string nm = temp();
                    o << "    " << T << " " << nm << " = " << zero << ";\n";
                    for (auto &t1 : terms) o << "    " << nm << " += " << t1 << ";\n";
                    cache.emplace_back(expr, nm);
                    name = nm;
                    return true;
                }
            }
            for (auto &c : cache)
                if (c.first == expr) {
                    name = c.second;
                    return true;
                }
            const std::string nm = temp();
            if (op.kind != kInter) ++chunk.values;
            (op.kind != kInter ? ld : o) << "    const " << T << " " << nm << " = " << expr << ";\n";
            cache.emplace_back(expr, nm);
            name = nm;
            return true;
        };
        for (uint32_t r = 0; r < nreg; ++r) {
            const uint32_t cst = pdep(r, RB);
            std::string va, vb;
            if (!value(0, cst, va) || !value(1, cst, vb)) return false;
            o << "    x" << s << "_" << r << " = " << (fp64 ? "fma(" : "fmaf(") << va << ", " << vb << ", x" << s << "_" << r
              << ");\n";
        }
        chunk.loads = ld.str();
        chunk.body = o.str();
        out.push_back(chunk);
    }
    std::ostringstream o;
    const int sh = fp64 ? st.a.cexp + st.b.cexp : rs ? -rs->shift[s] : 0;
    if (!dyn) {
        if (sh != 0)
            for (uint32_t r = 0; r < nreg; ++r)
                o << "    x" << s << "_" << r << " = " << (fp64 ? "ldexp(x" : "ldexpf(x") << s << "_" << r << ", " << sh << ");\n";
        out.back().body += o.str();
        return true;
    }
    // Entries are >= 0 or NaN, and NaN-ignoring fmaxf over them equals the
    // generic kernel's running `x > m ? x : m` from 0 (max is exact and order
    // free); a tree of three-input maxima halves the instructions.
    std::vector<std::string> mx;
    for (uint32_t r = 0; r < nreg; ++r) {
        o << "    x" << s << "_" << r << " = ldexpf(x" << s << "_" << r << ", shift" << S << ");\n";
        mx.push_back("x" + S + "_" + std::to_string(r));
    }
    mx.push_back("0.f");
    int nm = 0;
    while (mx.size() > 1) {
        std::vector<std::string> nx;
        for (size_t i = 0; i < mx.size(); i += 3) {
            if (i + 1 >= mx.size()) {
                nx.push_back(mx[i]);
                continue;
            }
            const std::string t = "lmax" + S + "_" + std::to_string(nm++);
            o << "    const float " << t << " = ";
            if (i + 2 < mx.size())
                o << "fmaxf(fmaxf(" << mx[i] << ", " << mx[i + 1] << "), " << mx[i + 2] << ");\n";
            else
                o << "fmaxf(" << mx[i] << ", " << mx[i + 1] << ");\n";
            nx.push_back(t);
        }
        mx.swap(nx);
    }
    o << "    float m" << S << " = " << mx[0] << ";\n";
    o << "    m" << S << " = fmaxf(QP(m" << S << ", 177), m" << S << ");\n    m" << S << " = fmaxf(QP(m" << S << ", 78), m" << S
      << ");\n";
    o << "    const int e" << S << " = ea" << S << " + eb" << S << ";\n";
    out.back().body += o.str();
    return true;
}

// The chunks in order, each one's table values loaded as many chunks ahead as
// keeps at most `budget` of them in flight: at two waves per SIMD nothing else
// hides a load, and left to itself the compiler loads a chunk's values right
// in front of it, one wait per 60 multiply-adds.  The scheduling barriers keep
// the loads where they are put.  Measured with emit_reg_syndrome on the d=7
// plan: FP32 64.2 -> 55.0 us per 65,536 rows and 20.9 -> 15.0 us for one tile
// (budgets of 8 to 24 agree within 2%, 32 and more spill: 70 us), FP64 117 ->
// 99 us.  Two waves per SIMD (224 registers) then wait 22% of their time and
// issue a VALU instruction every 4.7 cycles, 86% of them multiply-adds; chains
// of those alone issue one every 2.7 cycles with two waves.
void emit_reg_chunks(std::ostringstream &o, const std::vector<RegChunk> &chunks, int budget) {
    size_t next = 0;
    int flight = 0;
    for (size_t i = 0; i < chunks.size(); ++i) {
        bool any = false;
        while (next < chunks.size() && (next <= i || flight + chunks[next].values <= budget)) {
            o << chunks[next].loads;
            any = any || chunks[next].values > 0;
            flight += chunks[next++].values;
        }
        if (any) o << "    __builtin_amdgcn_sched_barrier(0);\n";
        o << chunks[i].body;
        flight -= chunks[i].values;
    }
}

// Syndrome bits of row b as s0, s1, ..: words as wide as the rows' alignment
// allows, all loads at once (a load of its own per bit under `valid ? :` cost a
// branch and a wait each, 5 us of the d=7 kernel's 21 us for one tile).
void emit_reg_syndrome(std::ostringstream &o, const CompiledPlan &cp, const std::vector<char> &used) {
    const int nb = std::max(1, cp.n_syn);
    const int w = nb % 16 == 0 ? 16 : nb % 8 == 0 ? 8 : nb % 4 == 0 ? 4 : 1;
    const int words = (nb + 3) / 4;
    o << "    unsigned sw[" << words << "];\n";
    const char *bytes = "    {\n"
                        "#pragma unroll\n"
                        "      for (int i = 0; i < NBITS; ++i) sw[i >> 2] = (i & 3 ? sw[i >> 2] : 0u) | ((unsigned)row[i] << (8 * (i & 3)));\n"
                        "    }\n";
    if (w == 1) {
        o << bytes;
    } else {
        const char *type = w == 16 ? "uint4" : w == 8 ? "uint2" : "unsigned";
        o << "    if (((unsigned long long)syn & " << (w - 1) << "ull) == 0ull) {\n";
        for (int i = 0; i < nb / w; ++i) {
            o << "      const " << type << " w" << i << " = reinterpret_cast<const " << type << " *>(row)[" << i << "];\n";
            const char *part[4] = {".x", ".y", ".z", ".w"};
            for (int c = 0; c < w / 4; ++c) o << "      sw[" << i * (w / 4) + c << "] = w" << i << (w == 4 ? "" : part[c]) << ";\n";
        }
        o << "    } else\n" << bytes;
    }
    for (int j = 0; j < cp.n_syn; ++j)
        if (used[j]) o << "    const unsigned s" << j << " = (sw[" << j / 4 << "] >> " << 8 * (j % 4) << ") & 1u;\n";
}

// ---- inline FP64 re-check of the register-resident FP32 kernel ------------
//
// The rows a tile flags are re-contracted by its waves, one row per wave: a
// row's latency is what counts (a batch of more than a few hundred rows has
// one in its last tiles nearly always), so its table slices are fetched to LDS
// all at once and the steps need no workgroup barrier.  A workgroup of 256
// threads that stepped through one row with a barrier and a table load from L2
// per step took 8.5 us for a row of the d=7 code and 3.5 us at d=3; this takes
// 7.3 and under 1 us, and several rows of a tile run side by side (65,536 rows
// of d=3 with 1,002 of them re-checked: 13.6 -> 9.9 us).

// LDS a workgroup may spend on it (beyond it, the separate kernel runs instead);
// with the FP32 tables in LDS no more than they leave: the 130 KB of a d=7 plan
// and the 33 KB of its four rows do not fit a CU together.
constexpr size_t kInlineRecheckLds = 48 * 1024;

size_t reg_tab_bytes(const CompiledPlan &cp, const SpecCfg &cfg) {
    return cfg.tab_lds ? std::max<size_t>(1, cp.const_pool.size() + cp.sliced_pool.size()) * (cfg.fp64 ? 8 : 4) : 0;
}

// its count and list of flagged rows, each aligned to 16 bytes at most
size_t reg_list_bytes(const SpecCfg &cfg) { return 16 + round_up((size_t)cfg.threads / 4 * 4, 16); }

struct Recheck {
    bool tables = false;                  // table slices staged in LDS
    std::vector<std::array<int, 2>> at;   // per step: LDS entry of its operands' slices, -1 for intermediates
    int entries = 0;                      // doubles per row: intermediates, then slices
    int rows = 0;                         // rows at a time (0: not inline)
};

Recheck recheck_plan(const CompiledPlan &cp, const SpecCfg &cfg) {
    Recheck r;
    if (!cfg.reg || cfg.fp64 || cp.ws_entries <= 0) return r;
    int64_t top = cp.ws_entries;
    for (const StepDesc &st : cp.steps) {
        std::array<int, 2> at = {-1, -1};
        for (int side = 0; side < 2; ++side) {
            const OperandDesc &op = side ? st.b : st.a;
            if (op.kind == kInter) continue;
            at[side] = (int)top;
            top += int64_t(1) << op.rank;
        }
        r.at.push_back(at);
    }
    size_t room = kInlineRecheckLds;
    if (cfg.tab_lds) {
        const size_t held = round_up(reg_tab_bytes(cp, cfg), 16) + reg_list_bytes(cfg);
        room = std::min(room, (kCuLds - std::min(kCuLds, held)) / 16 * 16);
    }
    r.tables = (size_t)top * 8 <= room;
    const int64_t e = r.tables ? top : cp.ws_entries;
    if ((size_t)e * 8 > room) return r;
    r.entries = (int)e;
    r.rows = (int)std::min<size_t>((size_t)cfg.threads / 64, room / ((size_t)e * 8));
    return r;
}

// recheck64: one row by one wave, the generic FP64 kernel's arithmetic; and
// the flagged rows wave, wave + r.rows, .. of a tile.
void emit_recheck_fn(std::ostringstream &o, const CompiledPlan &cp, const Recheck &r) {
    const int nb = std::max(1, cp.n_syn);
    const size_t const_n = cp.const_pool.size();
    o << "__device__ __attribute__((noinline)) void recheck64(const unsigned char *__restrict__ row, long long b,\n"
         "    const double *__restrict__ tab, double *__restrict__ mar, int *__restrict__ cls,\n"
         "    unsigned char *__restrict__ ties, double tie_tol, __attribute__((address_space(3))) double * work) {\n"
         "  using T = double;\n  constexpr int GLOG = 0, NOUT = "
      << (1 << cp.n_out) << ";\n  const int c0 = threadIdx.x & 63;\n";
    // the row's bits, uniform over the wave
    for (int w = 0; w * 64 < nb; ++w)
        o << "  const unsigned long long m" << w << " = __ballot(c0 < " << std::min(64, nb - 64 * w) << " && (row[" << 64 * w
          << " + min(c0, " << std::min(64, nb - 64 * w) - 1 << ")] & 1));\n";
    auto base = [&](const OperandDesc &op) {
        if (op.kind == kConst) return "tab + " + std::to_string((long long)op.off);
        std::string v = "0u";
        for (int j = 0; j < op.nev; ++j)
            v += " | (((unsigned)(m" + std::to_string(op.ev_bit[j] / 64) + " >> " + std::to_string(op.ev_bit[j] % 64) + ") & 1u) << " +
                 std::to_string(j) + ")";
        return "tab + " + std::to_string((long long)(const_n + (size_t)op.off)) + " + ((" + v + ") << " +
               std::to_string(op.rank) + ")";
    };
    if (r.tables) {
        // slices in groups of loads small enough for registers
        std::ostringstream ld, stg;
        int n = 0;
        auto flush = [&]() {
            o << "  {\n" << ld.str() << stg.str() << "  }\n";
            ld.str("");
            stg.str("");
            n = 0;
        };
        for (size_t s = 0; s < cp.steps.size(); ++s)
            for (int side = 0; side < 2; ++side) {
                const OperandDesc &op = side ? cp.steps[s].b : cp.steps[s].a;
                if (r.at[s][side] < 0) continue;
                const int size = 1 << op.rank;
                ld << "    const double *t" << s << "_" << side << " = " << base(op) << ";\n";
                for (int i = 0; i < size; i += 64) {
                    const std::string nm = "d" + std::to_string(s) + "_" + std::to_string(side) + "_" + std::to_string(i);
                    ld << "    const double " << nm << " = t" << s << "_" << side << "["
                       << (size < 64 ? "min(c0, " + std::to_string(size - 1) + ")" : "c0 + " + std::to_string(i)) << "];\n";
                    stg << "    " << (size < 64 ? "if (c0 < " + std::to_string(size) + ") " : "") << "work["
                        << r.at[s][side] + i << " + c0] = " << nm << ";\n";
                    ++n;
                }
                if (n >= 32) flush();
            }
        if (n) flush();
    }
    const char *sync = "  __threadfence_block();\n  __builtin_amdgcn_wave_barrier();\n";
    o << sync;
    for (size_t s = 0; s < cp.steps.size(); ++s) {
        const StepDesc &st = cp.steps[s];
        o << "  { // step " << s << "\n";
        for (int side = 0; side < 2; ++side) {
            const OperandDesc &op = side ? st.b : st.a;
            o << "    const auto p" << (side ? "b" : "a") << " = ";
            if (op.kind == kInter) o << "work + " << (long long)op.off << ";\n";
            else if (r.tables) o << "work + " << r.at[s][side] << ";\n";
            else o << base(op) << ";\n";
        }
        o << "    const auto pc = work + " << (long long)st.c_off << ";\n";
        emit_outputs(o, st, 64, 4, true);
        o << "  }\n" << sync;
    }
    o << "  if (c0 == 0) {\n"
         "    double best = 0, second = -1;\n"
         "    int bi = 0;\n"
         "    for (int j = 0; j < NOUT; ++j) {\n"
         "      const double x = work["
      << (long long)cp.root_off << " + j];\n"
         "      if (mar) mar[b * NOUT + j] = x;\n"
         "      if (j == 0 || x > best) {\n"
         "        if (j > 0) second = best;\n"
         "        best = x;\n"
         "        bi = j;\n"
         "      } else if (x > second) {\n"
         "        second = x;\n"
         "      }\n"
         "    }\n"
         "    if (cls) cls[b] = bi;\n"
         "    const bool low = NOUT > 1 && second >= 0 && best - second <= tie_tol * best;\n"
         "    if (ties) ties[b] = low ? 1 : 0;\n"
         "  }\n" << sync << "}\n\n";
    // LDS by its own address space (a generic pointer means flat loads and 182
    // registers instead of 136 at d=7); the loop stays outside the call: inside, its address arithmetic takes
    // registers (d=7: 248) that the call has to save
    o << "__device__ __forceinline__ void recheck64(const unsigned char *syn, int nf, const int *flagged, int wave,\n"
         "    const double *tab, double *mar, int *cls, unsigned char *ties, double tie_tol, __attribute__((address_space(3))) double * work) {\n"
         "  for (int i = wave; i < nf; i += " << r.rows << ")\n"
         "    recheck64(syn + (long long)flagged[i] * " << nb << ", (long long)flagged[i], tab, mar, cls, ties, tie_tol, work);\n"
         "}\n\n";
}

std::string reg_source(const CompiledPlan &cp, const SpecCfg &cfg, std::string &err) {
    RegPlan rp;
    if (!reg_plan(cp, rp)) {
        err = rp.err;
        return "";
    }
    const size_t const_n = cp.const_pool.size();
    const size_t tab_n = cp.const_pool.size() + cp.sliced_pool.size();
    const int G = cfg.threads / 4;
    const int nout = 1 << cp.n_out;
    const bool fp64 = cfg.fp64;
    const char *T = fp64 ? "double" : "float";
    std::ostringstream o;
    o << "// plan-specialised " << (fp64 ? "FP64" : "FP32")
      << " TNMMAP kernel, one syndrome per quad of lanes, tensors in registers (generated)\n";
    RegScale rsc;
    bool stat = false;
    if (!fp64 && !cfg.dyn) {
        std::string why;
        stat = reg_static_scales(cp, rp, rsc, why);
        if (stat)
            o << "// static exponents: root exponent " << rsc.e_root << ", FP64 re-check below 2^"
              << (int)std::ceil(rsc.theta) << " (true units)\n";
        else
            o << "// static scaling not applicable (" << why << "): per-step scaling\n";
    }
    const bool dyn = !fp64 && !stat;
    if (fp64)
        o << "#define QP(x, c) __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), (c), 0xf, 0xf, false), "
             "__builtin_amdgcn_mov_dpp(__double2loint(x), (c), 0xf, 0xf, false))\n";
    else
        o << "#define QP(x, c) __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), (c), 0xf, 0xf, false))\n";
    const Recheck rck = recheck_plan(cp, cfg);
    const bool inl = rck.rows > 0;
    // a call of its own, so that its registers do not crowd the FP32 program's
    if (inl) emit_recheck_fn(o, cp, rck);
    o << "extern \"C\" __global__ void __launch_bounds__(" << cfg.threads;
    if (cfg.waves > 0) o << ", " << cfg.waves;
    o << ") " << spec_kernel_name(cfg) << "(\n"
         "    const unsigned char *__restrict__ syn, long long n, const int *__restrict__ list,\n"
         "    const int *__restrict__ list_count, const " << T << " *__restrict__ gtab, double *__restrict__ mar,\n"
         "    int *__restrict__ cls, unsigned char *__restrict__ ties, int *__restrict__ rl,\n"
         "    int *__restrict__ rcount, long long rcap, double tie_tol, double recheck_tol, " << T
      << " *__restrict__ gslab,\n"
         "    int nseg, int segcap, const double *__restrict__ gtab64) {\n";
    o << "  constexpr int G = " << G << ", NBITS = " << std::max(1, cp.n_syn) << ", NOUT = " << nout << ";\n";
    o << "  (void)gslab; (void)nseg; (void)segcap; (void)gtab64;\n";
    o << "  __shared__ int seg_n;\n";
    if (inl) {
        // rows this tile flags for the FP64 re-check, done by the whole
        // workgroup at the end of the tile
        o << "  __shared__ int flagged[G];\n";
        o << "  __shared__ double work64[" << rck.rows << "][" << rck.entries << "];\n"
             "  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);\n";
    }
    if (cfg.tab_lds) {
        o << "  __shared__ " << T << " tab[" << std::max<size_t>(1, tab_n) << "];\n";
        o << "  for (int i = threadIdx.x; i < " << tab_n << "; i += " << cfg.threads << ") tab[i] = gtab[i];\n";
        o << "  __syncthreads();\n";
    } else {
        o << "  const " << T << " *tab = gtab;\n";
    }
    // Re-check list in per-tile segments: tile t's flagged rows go to
    // rl[t * rcap ..] and their number to rcount[t], written by every tile
    // the launch may own (those beyond a listed count write 0), so the list
    // needs no clearing between calls.
    o << "  const int q = threadIdx.x & 3;\n"
         "  const long long count = list ? (long long)(*list_count) : n;\n"
         "  const long long ntiles = (count + G - 1) / G;\n"
         "  const long long nseg_all = (n + G - 1) / G;\n"
         "  for (long long t = blockIdx.x; t < nseg_all; t += gridDim.x) {\n"
         "   if (threadIdx.x == 0) seg_n = 0;\n"
         "   __syncthreads();\n"
         "   if (t < ntiles) {\n"
         "    const long long qi = t * G + (threadIdx.x >> 2);\n"
         "    const bool valid = qi < count;\n"
         "    // lanes beyond the last row read it again and store nothing\n"
         "    const long long qc = valid ? qi : count - 1;\n"
         "    const long long b = list ? (long long)list[qc] : qc;\n"
         "    const unsigned char *row = syn + b * NBITS;\n";
    std::vector<char> used(std::max(1, cp.n_syn), 0);
    for (const StepDesc &st : cp.steps)
        for (const OperandDesc *op : {&st.a, &st.b})
            if (op->kind == kSliced)
                for (int j = 0; j < op->nev; ++j) used[op->ev_bit[j]] = 1;
    emit_reg_syndrome(o, cp, used);
    if (dyn) o << "    int lowf = 0;\n";
    std::vector<RegChunk> chunks;
    for (int s = 0; s < (int)cp.steps.size(); ++s)
        if (!emit_reg_step(chunks, cp, rp, s, const_n, fp64, stat ? &rsc : nullptr, err)) return "";
    emit_reg_chunks(o, chunks, fp64 ? kPrefetch64 : kPrefetch32);
    // every lane gathers the root's entries; the quad's lane 0 finishes the row
    const RLay &LR = rp.lay[rp.root];
    const std::vector<int> RR = reg_bits(LR, cp.steps[rp.root].rc);
    o << "    " << T << " rv[NOUT];\n";
    for (int j = 0; j < nout; ++j) {
        int src[4];
        for (int d = 0; d < 4; ++d) {
            src[d] = 0;
            for (int t = 0; t < 2; ++t) {
                const int bit = LR.pos[t] >= 0 ? ((j >> LR.pos[t]) & 1) : ((d >> t) & 1);
                src[d] |= bit << t;
            }
        }
        const int ctrl = quad_ctrl(src);
        const std::string nm = "x" + std::to_string(rp.root) + "_" + std::to_string(pext((uint32_t)j, RR));
        o << "    rv[" << j << "] = " << (ctrl == kIdentityCtrl ? nm : "QP(" + nm + ", " + std::to_string(ctrl) + ")") << ";\n";
    }
    o << "    if (q == 0 && valid) {\n"
         "      const int e = "
      << (fp64 ? std::string("0") : stat ? std::to_string(rsc.e_root) : "e" + std::to_string(rp.root)) << ";\n"
         "      " << T << " best = 0, second = -1;\n"
         "      int bi = 0;\n"
         "      for (int j = 0; j < NOUT; ++j) {\n"
         "        const " << T << " x = rv[j];\n"
         "        if (mar) mar[b * NOUT + j] = ldexp((double)x, e);\n"
         "        if (j == 0 || x > best) {\n"
         "          if (j > 0) second = best;\n"
         "          best = x;\n"
         "          bi = j;\n"
         "        } else if (x > second) {\n"
         "          second = x;\n"
         "        }\n"
         "      }\n"
         "      if (cls) cls[b] = bi;\n"
         "      const bool low = NOUT > 1 && second >= 0 && (double)(best - second) <= tie_tol * (double)best;\n"
         "      if (ties) ties[b] = low ? 1 : 0;\n";
    std::string low = "lowf != 0";
    if (stat) {
        // the root maximum in stored units against 2^(theta - e_root)
        const double lim = std::ceil(rsc.theta - rsc.e_root);
        char buf[64];
        std::snprintf(buf, sizeof(buf), "%.17g", lim < -1074 ? 0.0 : std::ldexp(1.0, (int)std::min(lim, 1000.0)));
        low = std::string("(double)best < ") + buf;
    }
    if (fp64)
        o << "      (void)recheck_tol;\n";
    else if (inl)
        o << "      {\n"
             "        const bool rc = !(best > 0) || " << low << " ||\n"
             "                        (NOUT > 1 && second >= 0 && (double)(best - second) <= recheck_tol * (double)best);\n"
             "        if (rc) flagged[atomicAdd(&seg_n, 1)] = (int)b;\n"
             "      }\n";
    else
        o << "      if (rl) {\n"
             "        const bool rc = !(best > 0) || " << low << " ||\n"
             "                        (NOUT > 1 && second >= 0 && (double)(best - second) <= recheck_tol * (double)best);\n"
             "        if (rc) {\n"
             "          const int slot = atomicAdd(&seg_n, 1);\n"
             "          if (slot < rcap) rl[t * rcap + slot] = (int)b;\n"
             "        }\n"
             "      }\n";
    o << "    }\n"
         "    }\n"
         "   }\n"
         "   __syncthreads();\n";
    if (inl)
        // at most G flagged rows (one per valid row of the tile)
        o << "   const int nf = seg_n;\n"
             "   if (wave < "
          << rck.rows << ") recheck64(syn, nf, flagged, wave, gtab64, mar, cls, ties, tie_tol,\n"
             "      (__attribute__((address_space(3))) double *)work64[wave]);\n"
             "   if (threadIdx.x == 0 && rcount) rcount[t] = nf;\n"
             "   __syncthreads();\n";
    else
        o << "   if (threadIdx.x == 0 && rcount) rcount[t] = min(seg_n, (int)rcap);\n";
    o << "  }\n"
         "}\n";
    return o.str();
}

}  // namespace

bool spec_reg_inline_recheck(const CompiledPlan &cp, const SpecCfg &cfg) {
    return recheck_plan(cp, cfg).rows > 0;
}

size_t spec_lds_bytes(const CompiledPlan &cp, const SpecCfg &cfg) {
    if (cfg.reg) {
        const Recheck r = recheck_plan(cp, cfg);
        const size_t tab = reg_tab_bytes(cp, cfg);
        if (r.rows == 0) return tab + 4;   // and the tile's count of flagged rows
        return round_up(tab, 16) + reg_list_bytes(cfg) + round_up((size_t)r.rows * r.entries * 8, 16);
    }
    return layout(cp, cfg).total;
}

bool spec_reg_supported(const CompiledPlan &cp, std::string *why) {
    RegPlan rp;
    const bool ok = reg_plan(cp, rp);
    if (!ok && why) *why = rp.err;
    return ok;
}

void spec_reg_prepare(CompiledPlan &cp) {
    cp.reg_lay.clear();
    cp.reg_checked = false;
    RegPlan rp;
    const bool ok = reg_plan(cp, rp);
    if (ok)
        for (const RLay &L : rp.lay) {
            cp.reg_lay.push_back(L.pos[0]);
            cp.reg_lay.push_back(L.pos[1]);
        }
    cp.reg_err = ok ? std::string() : rp.err;
    cp.reg_checked = true;
}

int spec_reg_peak(const CompiledPlan &cp) {
    RegPlan rp;
    reg_plan(cp, rp);
    return rp.peak;
}

size_t spec_slab_entries(const CompiledPlan &cp, const SpecCfg &cfg) {
    return cfg.slab ? (size_t)std::max<int64_t>(1, cp.ws_entries) << cfg.glog : 0;
}

namespace {

// `opaque`: hide the thread id from the compiler, so that nothing computed
// from it is moved out of the loop that calls the function.
// One tile of G syndromes (rows b0.., or list entries b0..) through the
// whole step program, as a device function: the body of the generic fused
// kernel's tile with every descriptor value substituted.  Starts and ends
// with a workgroup barrier.
void emit_tile_fn(std::ostringstream &o, const CompiledPlan &cp, const SpecCfg &cfg, const std::string &name,
                  bool opaque = false) {
    const Layout L = layout(cp, cfg);
    const size_t const_n = cp.const_pool.size();
    const int nsteps = (int)cp.steps.size();
    const char *tn = cfg.fp64 ? "double" : "float";
    o << "__device__ __forceinline__ void " << name << "(\n"
      << "    const unsigned char *__restrict__ syn, long long count, const int *__restrict__ list, long long b0,\n"
      << "    const " << tn << " *__restrict__ tab, double *__restrict__ mar, int *__restrict__ cls,\n"
      << "    unsigned char *__restrict__ ties, int *rl, int *rcount, long long rcap, double tie_tol,\n"
      << "    double recheck_tol, unsigned char *smem, " << tn << " *__restrict__ slabw, unsigned tag_base) {\n";
    o << "  using T = " << tn << ";\n";
    o << "  constexpr int G = " << (1 << cfg.glog) << ", GLOG = " << cfg.glog << ", NT = " << cfg.threads
      << ", CSTEP = " << (cfg.threads >> cfg.glog) << ", NBITS = " << std::max(1, cp.n_syn) << ", NOUT = "
      << (1 << cp.n_out) << ", NSLOTS = " << std::max(1, cp.n_slots) << ", RED = " << L.red << ";\n  (void)RED;\n";
    const Places places = slab_places(cp, cfg);
    if (cfg.slab)
        o << "  T *work = slabw;\n  T *lwork = reinterpret_cast<T *>(smem + " << L.work << ");\n  (void)lwork;\n";
    else
        o << "  T *work = reinterpret_cast<T *>(smem + " << L.work << ");\n";
    if (!cfg.fp64) {
        o << "  unsigned long long *mx = reinterpret_cast<unsigned long long *>(smem + " << L.mx << ");\n";
        o << "  int *ex = reinterpret_cast<int *>(smem + " << L.ex << ");\n";
        o << "  int *lowf = reinterpret_cast<int *>(smem + " << L.low << ");\n";
    }
    o << "  unsigned char *synl = smem + " << L.syn << ";\n";
    o << "  int tid = threadIdx.x;\n";
    if (opaque) o << "  asm volatile(\"\" : \"+v\"(tid));\n";
    o << "  const int g = tid & (G - 1);\n  const int c0 = tid >> GLOG;\n"
         "  const int lane = tid & 63;\n  (void)lane; (void)c0; (void)tag_base; (void)rl; (void)rcount; (void)rcap;\n"
         "  (void)recheck_tol; (void)NSLOTS;\n";
    o << "  if (!list) {\n"
         "    const long long rows = min((long long)G, count - b0);\n"
         "    const unsigned char *src = syn + b0 * NBITS;\n"
         "    for (int i = tid; i < G * NBITS; i += NT) {\n"
         "      const int r = i / NBITS, bit = i - r * NBITS;\n"
         "      synl[(bit << GLOG) + r] = (r < rows) ? (src[i] & 1u) : 0u;\n"
         "    }\n"
         "  } else {\n"
         "    for (int i = tid; i < G * NBITS; i += NT) {\n"
         "      const int r = i / NBITS, bit = i - r * NBITS;\n"
         "      const long long q = b0 + r;\n"
         "      synl[(bit << GLOG) + r] = (q < count) ? (syn[(long long)list[q] * NBITS + bit] & 1u) : 0u;\n"
         "    }\n"
         "  }\n";
    if (!cfg.fp64)
        o << "  for (int i = tid; i < NSLOTS * G; i += NT) mx[i] = 0ull;\n"
             "  if (tid < G) lowf[tid] = 0;\n";
    o << "  __syncthreads();\n";
    for (int s = 0; s < nsteps; ++s)
        emit_step(o, cp.steps[s], s, const_n, cfg.threads >> cfg.glog, cfg.fp64, std::max(1, cfg.unroll),
                  ((cfg.mfma || cfg.mfma32) && !cfg.fp64) ? &cfg : nullptr, places, cfg.slab);
    o << "  if (tid < G) {\n"
         "    const long long q = b0 + tid;\n"
         "    if (q < count) {\n"
         "      const long long b = list ? (long long)list[q] : q;\n";
    if (cfg.fp64)
        o << "      const int e = 0;\n";
    else
        o << "      const int e = ex[" << cp.root_slot << " * G + g];\n";
    o << "      T best = 0, second = -1;\n"
         "      int bi = 0;\n"
         "      for (int j = 0; j < NOUT; ++j) {\n";
    int64_t root_lds = -1;
    for (int s = 0; s < nsteps; ++s)
        if (cp.steps[s].is_root) root_lds = places.lds[s];
    o << "        const T x = " << (root_lds >= 0 ? "lwork" : "work") << "[("
      << (long long)(root_lds >= 0 ? root_lds : cp.root_off) << " + j) * G + g];\n";
    o << "        if (mar) mar[b * NOUT + j] = ldexp((double)x, e);\n"
         "        if (j == 0 || x > best) {\n"
         "          if (j > 0) second = best;\n"
         "          best = x;\n"
         "          bi = j;\n"
         "        } else if (x > second) {\n"
         "          second = x;\n"
         "        }\n"
         "      }\n"
         "      if (cls) cls[b] = bi;\n"
         "      const bool low = NOUT > 1 && second >= 0 && (double)(best - second) <= tie_tol * (double)best;\n"
         "      if (ties) ties[b] = low ? 1 : 0;\n";
    if (!cfg.fp64)
        o << "      if (rl) {\n"
         "        const bool rc = !(best > 0) || lowf[tid] != 0 ||\n"
         "                        (NOUT > 1 && second >= 0 && (double)(best - second) <= recheck_tol * (double)best);\n"
         "        if (rc) {\n"
         "          const int slot = atomicAdd(rcount, 1);\n"
         "          if (slot < rcap) rl[slot] = (int)b;\n"
         "        }\n"
         "      }\n";
    o << "    }\n"
         "  }\n"
         "  __syncthreads();\n"
         "}\n\n";
}

std::string dbl(double x) {
    char buf[64];
    std::snprintf(buf, sizeof(buf), "%.17g", x);
    return buf;
}

// Types and helpers of the generated MFMA steps.
const char *kMfmaPrelude =
    "typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8;\n"
    "typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;\n"
    "typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;\n"
    "__device__ __forceinline__ unsigned short to_bf16(float f) {\n"
    "  const unsigned u = __float_as_uint(f);\n"
    "  return (unsigned short)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);\n"
    "}\n\n";

}  // namespace

bool spec_step_uses_mfma32(const StepDesc &st, const SpecCfg &cfg) {
    if (!cfg.mfma32 || cfg.mfma || cfg.fp64 || cfg.reg || cfg.glog != 0 || cfg.threads % 64 != 0) return false;
    if ((st.a.kind == kInter && st.a.nsingle) || (st.b.kind == kInter && st.b.nsingle)) return false;
    std::vector<int> aon, bon;
    mfma_side_bits(st, aon, bon);
    if (aon.size() >= 5 && bon.size() >= 5) return st.nk >= 1;   // 32 x 32 x 2
    return aon.size() >= 4 && bon.size() >= 4 && st.nk >= 2;      // 16 x 16 x 4
}

bool spec_plan_uses_mfma32(const CompiledPlan &cp, const SpecCfg &cfg) {
    for (const StepDesc &st : cp.steps)
        if (spec_step_uses_mfma32(st, cfg)) return true;
    return false;
}

double spec_mfma32_share(const CompiledPlan &cp, const SpecCfg &cfg) {
    double all = 0, gemm = 0;
    for (const StepDesc &st : cp.steps) {
        const double macs = std::ldexp(1.0, st.rc + st.nk);
        all += macs;
        if (spec_step_uses_mfma32(st, cfg)) gemm += macs;
    }
    return all > 0 ? gemm / all : 0;
}

bool spec_step_uses_mfma(const StepDesc &st, const SpecCfg &cfg) {
    if (!cfg.mfma || cfg.fp64 || cfg.glog != 0 || cfg.threads % 64 != 0) return false;
    if (st.nk < 4) return false;
    if ((st.a.kind == kInter && st.a.nsingle) || (st.b.kind == kInter && st.b.nsingle)) return false;
    const uint32_t am = source_mask(st.a), bm = source_mask(st.b);
    const uint32_t outm = (st.rc >= 32) ? 0xffffffffu : ((1u << st.rc) - 1u);
    return __builtin_popcount(am & ~bm & outm) >= 5 && __builtin_popcount(bm & ~am & outm) >= 5;
}

std::string spec_source(const CompiledPlan &cp, const SpecCfg &cfg) {
    if (cfg.reg) {
        std::string err;
        return reg_source(cp, cfg, err);
    }
    const Layout L = layout(cp, cfg);
    const int nsteps = (int)cp.steps.size();
    std::ostringstream o;
    o << "// plan-specialised " << (cfg.fp64 ? "FP64" : "FP32") << " TNMMAP kernel (generated)\n";
    if (cfg.mfma || cfg.mfma32) o << kMfmaPrelude;
    emit_tile_fn(o, cp, cfg, "tile");
    const char *tn = cfg.fp64 ? "double" : "float";
    const int G = 1 << cfg.glog;
    o << "extern \"C\" __global__ void __launch_bounds__(" << cfg.threads;
    if (cfg.waves > 0) o << ", " << cfg.waves;
    o << ") " << spec_kernel_name(cfg) << "(\n"
      << "    const unsigned char *__restrict__ syn, long long n, const int *__restrict__ list,\n"
      << "    const int *__restrict__ list_count, const " << tn << " *__restrict__ gtab, double *__restrict__ mar,\n"
      << "    int *__restrict__ cls, unsigned char *__restrict__ ties, int *__restrict__ rl,\n"
      << "    int *__restrict__ rcount, long long rcap, double tie_tol, double recheck_tol, " << tn
      << " *__restrict__ gslab, int nseg, int segcap, const double *__restrict__ gtab64) {\n";
    o << "  (void)gtab64;\n";
    o << "  __shared__ __attribute__((aligned(16))) unsigned char smem[" << L.total << "];\n";
    if (cfg.tab_lds) {
        o << "  " << tn << " *tab = reinterpret_cast<" << tn << " *>(smem + " << L.tab << ");\n";
        o << "  for (int i = threadIdx.x; i < " << L.tab_entries << "; i += " << cfg.threads << ") tab[i] = gtab[i];\n";
    } else {
        o << "  const " << tn << " *tab = gtab;\n";
    }
    if (cfg.slab)
        o << "  " << tn << " *slabw = gslab + (unsigned long long)blockIdx.x * " << spec_slab_entries(cp, cfg) << "ull;\n";
    else
        o << "  " << tn << " *slabw = nullptr;\n";
    o << "  unsigned iter = 0;\n";
    // nseg > 0: the rows listed in per-tile segments (the register-resident
    // kernel's re-check list): segment w holds min(list_count[w], segcap)
    // rows at list[w * segcap ..]; each is decoded as row b0 of the syndrome
    // array (any row: a listed call's rows may lie beyond its count)
    o << "  if (nseg > 0) {\n"
         "    for (long long w = blockIdx.x; w < nseg; w += gridDim.x) {\n"
         "      const int c = min(list_count[w], segcap);\n"
         "      for (int e = 0; e < c; ++e, ++iter) {\n"
         "        const long long row = (long long)list[w * segcap + e];\n"
         "        tile(syn, row + 1, nullptr, row, tab, mar, cls, ties, rl, rcount, rcap, tie_tol, recheck_tol, smem, slabw,"
         " iter * " << nsteps << "u + 1u);\n"
         "      }\n"
         "    }\n"
         "    return;\n"
         "  }\n";
    o << "  const long long count = list ? (long long)(*list_count) : n;\n";
    o << "  const long long ntiles = (count + " << G - 1 << ") >> " << cfg.glog << ";\n";
    o << "  for (long long t = blockIdx.x; t < ntiles; t += gridDim.x, ++iter)\n";
    o << "    tile(syn, count, list, t << " << cfg.glog << ", tab, mar, cls, ties, rl, rcount, rcap, tie_tol, recheck_tol,"
         " smem, slabw, iter * " << nsteps << "u + 1u);\n";
    o << "}\n";
    return o.str();
}

std::string spec_map_source(const CompiledPlan &cp, int glog, int threads) {
    const int G = 1 << glog;
    const int ns = (int)cp.steps.size();
    const int words = (cp.n_vars + 31) / 32;
    const size_t work_b = (size_t)std::max<int64_t>(1, cp.ws_entries) * G * 8;
    const size_t arg_off = round_up(work_b, 16);
    const size_t syn_off = arg_off + round_up((size_t)std::max<int64_t>(1, cp.arg_entries) * G * 2, 16);
    const size_t total = round_up(syn_off + (size_t)std::max(1, cp.n_syn) * G, 16);
    std::ostringstream o;
    o << "// plan-specialised max-product (TNMAP) kernel (generated)\n";
    o << "extern \"C\" __global__ void __launch_bounds__(" << threads << ") tqec_map_spec(\n"
         "    const unsigned char *__restrict__ syn, long long n, const double *__restrict__ cpool,\n"
         "    const double *__restrict__ spool, unsigned char *__restrict__ config, int n_config,\n"
         "    double *__restrict__ logp) {\n";
    o << "  constexpr int G = " << G << ", GLOG = " << glog << ", NT = " << threads << ", CSTEP = " << (threads >> glog)
      << ", NBITS = " << std::max(1, cp.n_syn) << ", NV = " << cp.n_vars << ";\n";
    o << "  __shared__ __attribute__((aligned(16))) unsigned char smem[" << total << "];\n";
    o << "  double *work = reinterpret_cast<double *>(smem);\n";
    o << "  unsigned short *arg = reinterpret_cast<unsigned short *>(smem + " << arg_off << ");\n";
    o << "  unsigned char *synl = smem + " << syn_off << ";\n";
    o << "  const int tid = threadIdx.x, g = tid & (G - 1), c0 = tid >> GLOG;\n";
    o << "  const long long ntiles = (n + G - 1) >> GLOG;\n";
    o << "  for (long long t = blockIdx.x; t < ntiles; t += gridDim.x) {\n"
         "    const long long b0 = t << GLOG;\n"
         "    const long long rows = min((long long)G, n - b0);\n"
         "    const unsigned char *src = syn + b0 * NBITS;\n"
         "    for (int i = tid; i < G * NBITS; i += NT) {\n"
         "      const int r = i / NBITS, bit = i - r * NBITS;\n"
         "      synl[(bit << GLOG) + r] = (r < rows) ? (src[i] & 1u) : 0u;\n"
         "    }\n"
         "    __syncthreads();\n";
    // forward: every output keeps the first maximum over (k, sa, sb), as the generic kernel
    for (int s = 0; s < ns; ++s) {
        const StepDesc &st = cp.steps[s];
        const MapStep &ms = cp.map_steps[s];
        o << "    { // step " << s << ": rank " << st.rc << ", eliminated " << (st.nk + st.a.nsingle + st.b.nsingle)
          << "\n";
        const char *nm[2] = {"pa", "pb"};
        for (int side = 0; side < 2; ++side) {
            const OperandDesc &op = side ? st.b : st.a;
            if (op.kind == kInter) {
                o << "      const double *" << nm[side] << " = work + (" << (long long)op.off << "ll << GLOG) + g;\n";
            } else if (op.kind == kConst) {
                o << "      const double *" << nm[side] << " = cpool + " << (long long)op.off << ";\n";
            } else {
                o << "      unsigned v" << nm[side] << " = 0u;\n";
                for (int j = 0; j < op.nev; ++j)
                    o << "      v" << nm[side] << " |= (unsigned)synl[(" << op.ev_bit[j] << " << GLOG) + g] << " << j
                      << ";\n";
                o << "      const double *" << nm[side] << " = spool + " << (long long)op.off << " + ((long long)v"
                  << nm[side] << " << " << op.rank << ");\n";
            }
        }
        auto ld = [&](const OperandDesc &op, const char *base, const std::string &idx) {
            return op.kind == kInter ? std::string(base) + "[(" + idx + ") << GLOG]" : std::string(base) + "[" + idx + "]";
        };
        const int cexp = st.a.cexp + st.b.cexp;
        o << "      for (int c = c0; c < " << (1 << st.rc) << "; c += CSTEP) {\n";
        o << "        const unsigned ar = " << subst_c(gather_expr(st.a), "(unsigned)c") << ";\n";
        o << "        const unsigned br = " << subst_c(gather_expr(st.b), "(unsigned)c") << ";\n";
        o << "        double best = -1.0;\n        unsigned bi = 0u;\n";
        o << "        for (unsigned k = 0; k < " << (1u << st.nk) << "u; ++k)\n";
        o << "          for (unsigned qa = 0; qa < " << (1u << st.a.nsingle) << "u; ++qa) {\n";
        o << "            const double va = "
          << ld(st.a, "pa", "ar | (qa << " + std::to_string(st.a.sshift) + ") | (k << " + std::to_string(st.a.kshift) + ")")
          << ";\n";
        o << "            for (unsigned qb = 0; qb < " << (1u << st.b.nsingle) << "u; ++qb) {\n";
        o << "              const double vb = "
          << ld(st.b, "pb", "br | (qb << " + std::to_string(st.b.sshift) + ") | (k << " + std::to_string(st.b.kshift) + ")")
          << ";\n";
        o << "              const double v = va * vb;\n";
        o << "              if (v > best) {\n                best = v;\n                bi = k | (qa << " << st.nk
          << ") | (qb << " << (st.nk + st.a.nsingle) << ");\n              }\n";
        o << "            }\n          }\n";
        if (cexp != 0) o << "        best = ldexp(best, " << cexp << ");\n";
        o << "        work[((" << (long long)st.c_off << "ll + c) << GLOG) + g] = best;\n";
        o << "        arg[((" << (long long)ms.arg_off << "ll + c) << GLOG) + g] = (unsigned short)bi;\n";
        o << "      }\n    }\n    __syncthreads();\n";
    }
    // backtrace: one thread per syndrome, from the root down, labels as constants
    o << "    if (tid < G && b0 + tid < n) {\n";
    o << "      unsigned as[" << std::max(1, words) << "];\n";
    o << "      #pragma unroll\n      for (int w = 0; w < " << std::max(1, words) << "; ++w) as[w] = 0u;\n";
    for (int s = ns - 1; s >= 0; --s) {
        const MapStep &ms = cp.map_steps[s];
        const int32_t *L = cp.map_labels.data() + ms.off;
        o << "      {\n        unsigned c = 0u;\n";
        for (int j = 0; j < ms.nc; ++j)
            o << "        c |= ((as[" << (L[j] >> 5) << "] >> " << (L[j] & 31) << ") & 1u) << " << j << ";\n";
        o << "        const unsigned rec = arg[((" << (long long)ms.arg_off << "ll + c) << GLOG) + tid];\n";
        const int ne = ms.nk + ms.nsa + ms.nsb;
        for (int j = 0; j < ne; ++j) {
            const int l = L[ms.nc + j];
            o << "        as[" << (l >> 5) << "] |= ((rec >> " << j << ") & 1u) << " << (l & 31) << ";\n";
        }
        o << "      }\n";
    }
    o << "      const long long b = b0 + tid;\n";
    o << "      #pragma unroll\n      for (int v = 0; v < NV; ++v)\n"
         "        if (v < n_config) config[b * n_config + v] = (unsigned char)((as[v >> 5] >> (v & 31)) & 1u);\n";
    o << "      if (logp) logp[b] = log(work[(" << (long long)cp.root_off << "ll << GLOG) + tid]);\n";
    o << "    }\n    __syncthreads();\n  }\n}\n";
    return o.str();
}

namespace {

// Largest table set that a workgroup of the wave max-product kernel copies to LDS.
constexpr size_t kMapTabLds = 16 * 1024;

// Records of a wave at most (64 bits each, two vector registers for 64 of
// them), and blocks of outputs of one step among which the backtrace selects.
constexpr int kMapMaxRecords = 512, kMapMaxBlocks = 8;

// Records of a step: bits eliminated times 64-entry blocks of (output, syndrome).
int map_blocks(const StepDesc &st, int glog) { return std::max(1, (1 << st.rc) >> (6 - glog)); }

struct MapWaveLayout {
    size_t tab = 0;                      // bytes at the start of the workgroup's LDS
    size_t syn = 0, total = 0;           // per wave
    std::vector<int> rec_at;             // first 64-bit record of each step
    int nrec = 0, max_blocks = 1;
};

MapWaveLayout map_wave_layout(const CompiledPlan &cp, int glog) {
    MapWaveLayout L;
    const size_t tab = (cp.const_pool.size() + cp.sliced_pool.size()) * 8;
    if (tab <= kMapTabLds) L.tab = round_up(tab, 16);
    for (const StepDesc &st : cp.steps) {
        L.rec_at.push_back(L.nrec);
        L.nrec += map_blocks(st, glog) * (st.nk + st.a.nsingle + st.b.nsingle);
        L.max_blocks = std::max(L.max_blocks, map_blocks(st, glog));
    }
    const size_t words = (size_t)(cp.n_vars + 31) / 32;
    L.syn = round_up(((size_t)std::max<int64_t>(1, cp.ws_entries) * 8) << glog, 16);
    // the syndrome's bytes, later the configuration's words
    L.total = round_up(L.syn + (std::max((size_t)std::max(1, cp.n_syn), words * 4) << glog), 16);
    return L;
}

}  // namespace

// A d=5 plan has 75 steps of 9 outputs on average: a workgroup tile spends its
// time on 75 barriers, a table load from global memory before each, and a
// backtrace by 16 of 256 threads.  A wave takes as many syndromes as leave its
// lanes an output each on average; fewer where eight waves would not share the
// LDS.  us, workgroup tile -> G = 2 / 4 / 8 per wave: 16,384 rows 47 -> 52 / 29
// / 23, 65,536 rows 162 -> 170 / 108 / 82 (d=3, 65,536 rows, G = 4 / 8 / 16: 23
// / 14 / 11).  Three waves per SIMD, and the lane id hidden in the group loop:
// the compiler otherwise moves the address arithmetic of all steps out of it,
// and with all the registers it wants for that (one wave per SIMD) the 23 us
// are 31; a d=7 plan takes 151 us per 16,384 rows instead of 215.
bool spec_map_wave_cfg(const CompiledPlan &cp, size_t lds_limit, int &glog, int &waves) {
    if (cp.steps.empty()) return false;
    int64_t outputs = 0;
    for (const StepDesc &st : cp.steps) {
        outputs += int64_t(1) << st.rc;
        if (st.nk + st.a.nsingle + st.b.nsingle > 16 || st.rc > 16) return false;
    }
    const int64_t mean = outputs / (int64_t)cp.steps.size();
    for (glog = 4; glog > 0 && (mean << glog) > 80; --glog) {}
    for (;; --glog) {
        if (glog < 0) return false;
        const MapWaveLayout L = map_wave_layout(cp, glog);
        if (L.nrec > kMapMaxRecords || L.max_blocks > kMapMaxBlocks) continue;
        for (waves = 4; waves >= 1; waves >>= 1)
            if (8 / waves * (L.tab + (size_t)waves * L.total) <= lds_limit) return true;
    }
}

std::string spec_map_wave_source(const CompiledPlan &cp, int glog, int waves) {
    const int G = 1 << glog, lanes = 64 >> glog, cl = 6 - glog, nt = waves * 64;
    const int ns = (int)cp.steps.size();
    const int words = (cp.n_vars + 31) / 32;
    const size_t const_n = cp.const_pool.size(), tab_n = const_n + cp.sliced_pool.size();
    const MapWaveLayout W = map_wave_layout(cp, glog);
    std::ostringstream o;
    o << "// plan-specialised max-product (TNMAP) kernel, a wave per " << G << " syndromes (generated)\n";
    o << "extern \"C\" __global__ void __launch_bounds__(" << nt << ", 3) tqec_map_spec(\n"
         "    const unsigned char *__restrict__ syn, long long n, const double *__restrict__ cpool,\n"
         "    const double *__restrict__ spool, unsigned char *__restrict__ config, int n_config,\n"
         "    double *__restrict__ logp) {\n";
    o << "  constexpr int G = " << G << ", GLOG = " << glog << ", LANES = " << lanes << ", NBITS = " << cp.n_syn
      << ";\n";
    o << "  __shared__ __attribute__((aligned(16))) unsigned char smem[" << W.tab + (size_t)waves * W.total << "];\n";
    o << "  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);\n";
    o << "  unsigned char *mine = smem + " << W.tab << " + wave * " << W.total << ";\n"
         "  unsigned char *synl = mine + " << W.syn << ";\n"
         "  unsigned *cfgw = reinterpret_cast<unsigned *>(synl);\n";
    if (W.tab) {
        o << "  double *tab = reinterpret_cast<double *>(smem);\n"
             "  for (int i = threadIdx.x; i < " << const_n << "; i += " << nt << ") tab[i] = cpool[i];\n"
             "  for (int i = threadIdx.x; i < " << tab_n - const_n << "; i += " << nt << ") tab[" << const_n
          << " + i] = spool[i];\n"
             "  const double *tc = tab, *ts = tab + " << const_n << ";\n"
             "  __syncthreads();\n";
    } else {
        o << "  const double *tc = cpool, *ts = spool;\n";
    }
    const char *fence = "__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, \"wavefront\"); __builtin_amdgcn_wave_barrier();\n";
    o << "  const long long ntiles = (n + G - 1) >> GLOG;\n"
         "  for (long long t = (long long)blockIdx.x * " << waves << " + wave; t < ntiles; t += (long long)gridDim.x * "
      << waves << ") {\n"
         "    int lane = threadIdx.x & 63;\n"
         "    asm volatile(\"\" : \"+v\"(lane));   // keeps address arithmetic inside the loop\n"
         "    const int g = lane & (G - 1), c0 = lane >> GLOG;\n"
         "    double *work = reinterpret_cast<double *>(mine) + g;\n"
         "    const long long q = (t << GLOG) + g;\n"
         "    const bool valid = q < n;\n"
         "    // lanes beyond the last row read it again and store nothing\n"
         "    const long long b = valid ? q : n - 1;\n"
         "    for (int i = c0; i < NBITS; i += LANES) synl[(i << GLOG) + g] = syn[b * NBITS + i] & 1u;\n    " << fence;
    // arg-max records: uniform 64-bit words, a bit per (output, syndrome); the
    // compiler keeps those beyond the scalar registers in vector lanes
    for (int r = 0; r < W.nrec; ++r) o << "    unsigned long long r" << r << ";\n";
    for (int s = 0; s < ns; ++s) {
        const StepDesc &st = cp.steps[s];
        const int nb = st.nk + st.a.nsingle + st.b.nsingle;
        o << "    { // step " << s << ": rank " << st.rc << ", eliminated " << nb << "\n";
        for (int side = 0; side < 2; ++side) {
            const OperandDesc &op = side ? st.b : st.a;
            const char *nm = side ? "pb" : "pa";
            if (op.kind == kInter) {
                o << "      const double *" << nm << " = work + " << ((long long)op.off << glog) << ";\n";
            } else if (op.kind == kConst) {
                o << "      const double *" << nm << " = tc + " << (long long)op.off << ";\n";
            } else {
                o << "      unsigned v" << nm << " = 0u;\n";
                for (int j = 0; j < op.nev; ++j)
                    o << "      v" << nm << " |= (unsigned)synl[(" << op.ev_bit[j] << " << GLOG) + g] << " << j << ";\n";
                o << "      const double *" << nm << " = ts + " << (long long)op.off << " + (v" << nm << " << " << op.rank
                  << ");\n";
            }
        }
        // every output keeps the first maximum over (k, sa, sb), as the generic kernel
        const int nk = 1 << st.nk, na = 1 << st.a.nsingle, nbn = 1 << st.b.nsingle;
        const int terms = nk * (na + nbn), blocks = map_blocks(st, glog);
        const int cexp = st.a.cexp + st.b.cexp;
        const std::string ga = gather_expr(st.a), gb = gather_expr(st.b);
        const unsigned cmask = (1u << st.rc) - 1u;
        // outputs of a chunk: loads first, then comparisons, then stores
        const int chunk = std::max(1, std::min(blocks, 32 / std::max(1, terms)));
        const bool flat = terms <= 64;
        for (int x0 = 0; x0 < blocks; x0 += chunk) {
            const int x1 = std::min(blocks, x0 + chunk);
            o << "      {\n";
            for (int x = x0; x < x1; ++x) {
                const std::string X = std::to_string(x);
                o << "      const unsigned oc" << X << " = ((unsigned)c0 | " << ((unsigned)x << cl) << "u) & " << cmask
                  << "u;\n";
                o << "      const double *a" << X << " = pa + ((" << subst_c(ga, "oc" + X) << ")"
                  << (st.a.kind == kInter ? " << GLOG" : "") << ");\n";
                o << "      const double *b" << X << " = pb + ((" << subst_c(gb, "oc" + X) << ")"
                  << (st.b.kind == kInter ? " << GLOG" : "") << ");\n";
                o << "      double best" << X << " = -1.0;\n      unsigned bi" << X << " = 0u;\n";
                if (!flat) continue;
                for (int k = 0; k < nk; ++k) {
                    for (int qa = 0; qa < na; ++qa)
                        o << "      const double u" << X << "_" << k << "_" << qa << " = a" << X << "["
                          << ((((unsigned)qa << st.a.sshift) | ((unsigned)k << st.a.kshift))
                              << (st.a.kind == kInter ? glog : 0))
                          << "];\n";
                    for (int qb = 0; qb < nbn; ++qb)
                        o << "      const double w" << X << "_" << k << "_" << qb << " = b" << X << "["
                          << ((((unsigned)qb << st.b.sshift) | ((unsigned)k << st.b.kshift))
                              << (st.b.kind == kInter ? glog : 0))
                          << "];\n";
                }
            }
            for (int x = x0; x < x1; ++x) {
                const std::string X = std::to_string(x);
                if (flat) {
                    for (int k = 0; k < nk; ++k)
                        for (int qa = 0; qa < na; ++qa)
                            for (int qb = 0; qb < nbn; ++qb)
                                o << "      { const double v = u" << X << "_" << k << "_" << qa << " * w" << X << "_" << k
                                  << "_" << qb << "; if (v > best" << X << ") { best" << X << " = v; bi" << X << " = "
                                  << (unsigned)(k | (qa << st.nk) | (qb << (st.nk + st.a.nsingle))) << "u; } }\n";
                } else {
                    const auto idx = [&](const char *qn, const OperandDesc &op) {
                        return std::string("(((unsigned)") + qn + " << " + std::to_string(op.sshift) + ") | ((unsigned)k << " +
                               std::to_string(op.kshift) + "))" + (op.kind == kInter ? " << GLOG" : "");
                    };
                    o << "      for (int k = 0; k < " << nk << "; ++k)\n        for (int qa = 0; qa < " << na
                      << "; ++qa) {\n          const double va = a" << X << "[" << idx("qa", st.a) << "];\n"
                      << "          for (int qb = 0; qb < " << nbn << "; ++qb) {\n            const double v = va * b" << X
                      << "[" << idx("qb", st.b) << "];\n            if (v > best" << X << ") { best" << X << " = v; bi" << X
                      << " = (unsigned)k | ((unsigned)qa << " << st.nk << ") | ((unsigned)qb << " << st.nk + st.a.nsingle
                      << "); }\n          }\n        }\n";
                }
                if (cexp != 0) o << "      best" << X << " = ldexp(best" << X << ", " << cexp << ");\n";
            }
            for (int x = x0; x < x1; ++x) {
                const std::string X = std::to_string(x);
                o << "      work[(" << (long long)st.c_off << " + oc" << X << ") << GLOG] = best" << X << ";\n";
                for (int j = 0; j < nb; ++j)
                    o << "      r" << W.rec_at[s] + x * nb + j << " = __ballot((bi" << X << " >> " << j << ") & 1u);\n";
            }
            o << "      }\n";
        }
        o << "    }\n    " << fence;
    }
    // backtrace: every lane of a syndrome follows it, from the root down, with
    // a register per label; a step's record is bit (output, syndrome) of its block
    std::vector<char> known(std::max(1, cp.n_vars), 0);
    for (int s = ns - 1; s >= 0; --s) {
        const StepDesc &st = cp.steps[s];
        const MapStep &ms = cp.map_steps[s];
        const int32_t *lab = cp.map_labels.data() + ms.off;
        const int nb = st.nk + st.a.nsingle + st.b.nsingle, blocks = map_blocks(st, glog);
        if (!nb) continue;
        for (int j = 0; j < nb; ++j)
            if (!known[lab[ms.nc + j]]) {
                known[lab[ms.nc + j]] = 1;
                o << "    unsigned L" << lab[ms.nc + j] << " = 0u;\n";
            }
        o << "    {\n      unsigned c = 0u;\n";
        for (int j = 0; j < ms.nc; ++j)
            if (known[lab[j]]) o << "      c |= L" << lab[j] << " << " << j << ";\n";
        o << "      const unsigned at = ((c & " << lanes - 1 << "u) << GLOG) | (unsigned)g;\n";
        // 32-bit halves: no 64-bit shifts by a vector register (see mask_bit in
        // sampler_hip.hip)
        const bool low = (int64_t(1) << (st.rc + glog)) <= 32;
        for (int j = 0; j < nb; ++j)
            for (int x = 0; x < blocks; ++x) {
                const std::string r = "r" + std::to_string(W.rec_at[s] + x * nb + j);
                o << "      ";
                if (blocks > 1) o << "if ((c >> " << cl << ") == " << x << "u) ";
                o << "L" << lab[ms.nc + j] << " |= __builtin_amdgcn_ubfe(";
                if (low) o << "(unsigned)" << r;
                else o << "at < 32u ? (unsigned)" << r << " : (unsigned)(" << r << " >> 32)";
                o << ", at" << (low ? "" : " & 31u") << ", 1u);\n";
            }
        o << "    }\n";
    }
    for (int w = 0; w < words; ++w) {
        o << "    cfgw[" << (w << glog) << " + g] = 0u";
        for (int v = 32 * w; v < std::min(cp.n_vars, 32 * w + 32); ++v)
            if (known[v]) o << " | (L" << v << " << " << (v & 31) << ")";
        o << ";\n";
    }
    o << "    " << fence;
    o << "    if (valid)\n"
         "      for (int v = c0; v < n_config; v += LANES)\n"
         "        config[b * n_config + v] = (unsigned char)((cfgw[((v >> 5) << GLOG) + g] >> (v & 31)) & 1u);\n"
         "    if (valid && c0 == 0 && logp) logp[b] = log(work[" << ((long long)cp.root_off << glog) << "]);\n    "
      << fence << "  }\n}\n";
    return o.str();
}

size_t spec_mixed_lds_bytes(const std::vector<MixedSpecPlan> &plans) {
    size_t m = 16;
    for (const MixedSpecPlan &q : plans) {
        m = std::max(m, layout(*q.cp, q.f32).total);
        m = std::max(m, layout(*q.cp, q.f64).total);
    }
    return m;
}

std::string spec_mixed_source(const std::vector<MixedSpecPlan> &plans, int threads, size_t slab32_entries,
                              size_t slab64_entries, int cus) {
    std::ostringstream o;
    o << "// mixed-code kernel: plan-specialised tiles of " << plans.size() << " plans (generated)\n";
    bool any_mfma = false;
    for (const MixedSpecPlan &q : plans) any_mfma = any_mfma || q.f32.mfma || q.f32.mfma32;
    if (any_mfma) o << kMfmaPrelude;
    // the layouts of the host's batch table, header and counters
    o << "struct MBatch { const unsigned char *syn; double *mar; int *cls; unsigned char *tie; long long n;\n"
         "                long long tile0; int plan; int glog; };\n"
         "struct MHeader { int nbatches; int pad; long long ntiles; };\n"
         "struct MCounters { unsigned long long next_tile; unsigned long long next_recheck; int rl_count; int pad;\n"
         "                   unsigned long long t_start; };\n\n";
    for (size_t i = 0; i < plans.size(); ++i) {
        emit_tile_fn(o, *plans[i].cp, plans[i].f32, "p" + std::to_string(i) + "_f32", true);
        emit_tile_fn(o, *plans[i].cp, plans[i].f64, "p" + std::to_string(i) + "_f64", true);
    }
    // As many workgroups of 256 threads per CU as their LDS allows, three at
    // most.  Left to itself the compiler takes registers for one, once it has
    // moved every plan's address arithmetic out of the tile loop (the tile
    // functions hide their thread id to keep it inside).  Held to three it
    // spills where a plan runs from a slab on MFMA (24 registers, 100 B per
    // lane; none in mixes of LDS plans), which still pays: 48 batches, 22,185
    // rows of five codes, a third of them toric L=3, 557 us; held to two 720,
    // to one 916 (24 batches, 6,783 rows with 76 of toric L=3: 59, 62 and 58).
    // A d=7 plan's tiles leave room for two (67 KB): 24 batches of 3,000 rows
    // of six codes 1,158 us, and 1,863 held to three, which the compiler takes
    // for no bound at all.
    const size_t lds = spec_mixed_lds_bytes(plans) + kMixedStaticLds;
    const size_t wgs = threads == 256 ? std::max<size_t>(1, std::min<size_t>(3, kCuLds / lds)) : 1;
    o << "extern \"C\" __global__ void __launch_bounds__(" << threads << ", " << wgs
      << ") tqec_mixed_spec(\n"
         "    const MBatch *__restrict__ batches, const MHeader *__restrict__ hdr, MCounters *ctr,\n"
         "    unsigned long long *t_done, const float *const *tabs32, const double *const *tabs64, float *slab32,\n"
         "    double *slab64) {\n";
    o << "  __shared__ __attribute__((aligned(16))) unsigned char smem[" << spec_mixed_lds_bytes(plans) << "];\n";
    o << "  __shared__ long long grab;\n  __shared__ int loc_n;\n  __shared__ int loc_rows[64];\n";
    o << "  float *s32 = slab32 ? slab32 + (unsigned long long)blockIdx.x * " << slab32_entries << "ull : nullptr;\n";
    o << "  double *s64 = slab64 ? slab64 + (unsigned long long)blockIdx.x * " << slab64_entries << "ull : nullptr;\n";
    // few tiles: one workgroup per CU takes them, rather than any of three
    o << "  const int nb = hdr->nbatches;\n  const long long ntiles = hdr->ntiles;\n"
         "  if (ntiles <= "
      << 2 * cus << " && blockIdx.x >= " << cus << ") return;\n"
         "  unsigned tag = 1;\n  bool first = true;\n"
         "  if (threadIdx.x == 0) loc_n = 0;\n"
         "  for (;;) {\n"
         "    __syncthreads();\n"
         "    if (threadIdx.x == 0) grab = (long long)atomicAdd(&ctr->next_tile, 1ull);\n"
         "    __syncthreads();\n"
         "    const long long t = grab;\n"
         "    if (t >= ntiles) break;\n"
         "    if (first && threadIdx.x == 0) atomicMin(&ctr->t_start, (unsigned long long)wall_clock64());\n"
         "    first = false;\n"
         "    int lo = 0, hi = nb - 1;\n"
         "    while (lo < hi) {\n"
         "      const int mid = (lo + hi + 1) >> 1;\n"
         "      if (batches[mid].tile0 <= t) lo = mid; else hi = mid - 1;\n"
         "    }\n"
         "    const MBatch bt = batches[lo];\n"
         "    switch (bt.plan) {\n";
    for (size_t i = 0; i < plans.size(); ++i) {
        const MixedSpecPlan &q = plans[i];
        o << "    case " << i << ":\n      p" << i << "_f32(bt.syn, bt.n, nullptr, (t - bt.tile0) << " << q.f32.glog
          << ", tabs32[" << i << "], bt.mar, bt.cls, bt.tie, loc_rows, &loc_n, 64, " << dbl(q.tie_tol) << ", "
          << dbl(q.recheck_tol) << ", smem, s32, tag);\n      tag += " << q.cp->steps.size() << "u;\n      break;\n";
    }
    o << "    default: break;\n    }\n";
    o << "    const int nre = loc_n;\n"
         "    if (nre > 0) {\n"
         "      for (int e = 0; e < nre; ++e) {\n"
         "        const long long row = loc_rows[e];\n"
         "        switch (bt.plan) {\n";
    for (size_t i = 0; i < plans.size(); ++i) {
        const MixedSpecPlan &q = plans[i];
        o << "        case " << i << ":\n          p" << i << "_f64(bt.syn, bt.n, nullptr, row, tabs64[" << i
          << "], bt.mar, bt.cls, bt.tie, nullptr, nullptr, 0, " << dbl(q.tie_tol) << ", " << dbl(q.recheck_tol)
          << ", smem, s64, 1u);\n          break;\n";
    }
    o << "        default: break;\n        }\n"
         "      }\n"
         "      if (threadIdx.x == 0) {\n"
         "        atomicAdd(&ctr->rl_count, nre);\n"
         "        loc_n = 0;\n"
         "      }\n"
         "    }\n"
         "    if (threadIdx.x == 0) atomicMax(&t_done[lo], (unsigned long long)wall_clock64());\n"
         "  }\n"
         "}\n";
    return o.str();
}

}  // namespace tqec
