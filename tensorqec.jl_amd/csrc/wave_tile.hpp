// wave_tile.hpp — generic fused executor, one wavefront per group of
// G = 2^glog syndromes (G = 1, 2, 4, 8).
//
// The interpreter's time is latency: a step of a d=5 or d=7 plan is a few
// hundred multiply-adds, so what counts is how many dependent loads, barriers
// and iterations lie between one step and the next.  Here
//   * the step descriptors are 32 words each (WavePlan), copied to LDS once per
//     workgroup; a wave reads the next step's into one register per lane while
//     it works on this one and takes fields out with v_readlane;
//   * every table slice that a syndrome selects is copied to LDS before the
//     first step, all loads in flight at once, so the steps read LDS only;
//   * a wave owns its syndromes, so steps need no workgroup barrier, the scale
//     maximum is reduced with lane permutations, and no atomics are left;
//   * operand indexes are the bits of the output index moved about: the lane's
//     own six bits once per step, the others one XOR per output (Gray order),
//     and up to four outputs of four terms each are in flight.
// Every output entry is the same chain of multiply-adds, scale and maximum as
// in fused_tile, so results are bit-identical to it for any G.
#pragma once
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>
#include <vector>

#include "plan_compile.hpp"

namespace tqec {

constexpr int kWaveWords = 32;      // descriptor words of a step
constexpr int kWaveBits = 16;       // first word of the output bits' moves
constexpr int kWaveOpWords = 8;     // words of a staged operand
constexpr int kWaveMaxGlog = 3;

// Device form of a plan for wave_kernel: steps, staged operands, staged entries.
struct WavePlan {
    std::vector<uint32_t> desc;     // nsteps * kWaveWords, then nops * kWaveOpWords
    std::vector<uint32_t> ent;      // per staged entry: operand << 16 | index in the slice
    int nsteps = 0, nops = 0;
    int64_t mean_outputs = 0;       // output entries per step
    bool ok = false;
};

inline WavePlan wave_plan(const CompiledPlan &cp) {
    WavePlan w;
    int64_t at = cp.ws_entries;
    const int64_t const_n = (int64_t)cp.const_pool.size();
    if (at > 32768 || cp.n_syn >= 65535 || cp.n_slots > 65535 || cp.steps.empty()) return w;
    std::vector<uint32_t> ops;
    auto stage = [&](const OperandDesc &op) -> int64_t {
        if (op.kind == kInter) return op.off;
        uint32_t q[kWaveOpWords] = {};
        const int64_t base = op.kind == kConst ? op.off : const_n + op.off;
        q[0] = (uint32_t)base;
        q[1] = (uint32_t)op.rank;
        const int nev = op.kind == kSliced ? op.nev : 0;
        // selector bits that are not there read a bit that is always zero
        for (int j = 0; j < kMaxEv; ++j)
            q[2 + j / 2] |= (uint32_t)(j < nev ? op.ev_bit[j] : cp.n_syn) << (16 * (j & 1));
        const uint32_t id = (uint32_t)(ops.size() / kWaveOpWords);
        for (int64_t i = 0; i < (int64_t(1) << op.rank); ++i) w.ent.push_back(id << 16 | (uint32_t)i);
        ops.insert(ops.end(), q, q + kWaveOpWords);
        const int64_t r = at;
        at += int64_t(1) << op.rank;
        return r;
    };
    for (const StepDesc &st : cp.steps) {
        if (st.rc > kWaveWords - kWaveBits || st.nk > 15 || st.a.rank > 15 || st.b.rank > 15) return w;
        uint32_t d[kWaveWords] = {};
        const bool aw = st.a.kind == kInter, bw = st.b.kind == kInter;
        const int nsa = aw ? st.a.nsingle : 0, nsb = bw ? st.b.nsingle : 0;
        d[0] = (uint32_t)st.rc | (uint32_t)st.nk << 8 | (uint32_t)aw << 16 | (uint32_t)bw << 17;
        d[1] = (uint32_t)stage(st.a);
        d[2] = (uint32_t)stage(st.b);
        if (at > 32768 || ops.size() / kWaveOpWords > 65535) return w;
        d[3] = (uint32_t)st.c_off;
        d[4] = (uint32_t)st.a.kshift | (uint32_t)st.b.kshift << 8 | (uint32_t)nsa << 16 | (uint32_t)nsb << 24;
        d[5] = (uint32_t)st.a.sshift | (uint32_t)st.b.sshift << 8;
        d[6] = aw ? (uint32_t)st.a.slot : 0u;
        d[7] = bw ? (uint32_t)st.b.slot : 0u;
        d[8] = (uint32_t)st.c_slot;
        d[9] = (uint32_t)st.a.cexp;
        d[10] = (uint32_t)st.b.cexp;
        for (int t = 0; t < st.rc; ++t)
            d[kWaveBits + t] = gather_bits(1u << t, st.a) | gather_bits(1u << t, st.b) << 16;
        w.mean_outputs += int64_t(1) << st.rc;
        w.desc.insert(w.desc.end(), d, d + kWaveWords);
    }
    w.nsteps = (int)cp.steps.size();
    w.mean_outputs /= w.nsteps;
    w.nops = (int)(ops.size() / kWaveOpWords);
    w.desc.insert(w.desc.end(), ops.begin(), ops.end());
    if (w.ent.empty()) w.ent.push_back(0);
    w.ok = true;
    return w;
}

// Sizes the kernel and the host agree on.
struct WaveDims {
    int nsteps, nops, nent, ws, nslots, nbits, glog;
    __host__ __device__ int desc_bytes() const { return (nsteps * kWaveWords + nops * kWaveOpWords) * 4; }
    __host__ __device__ int vals() const { return ws + nent; }
    __host__ __device__ int wave_bytes(int elem) const {
        const int b = ((vals() * elem + (2 * nslots + nops) * 4) << glog) + ((nbits + 1) << glog);
        return (b + 15) & ~15;
    }
};

struct WaveArgs {
    WaveDims d;
    const uint32_t *desc;
    const uint32_t *ent;
    const void *tab;            // constant pool, then the sliced pool
    const uint8_t *syn;         // [n][nbits]
    int64_t n;
    int nout;
    int root_off, root_slot;
    const int32_t *list;        // optional: syndrome ids to process
    const int32_t *list_count;
    double *marginals;
    int32_t *classes;
    uint8_t *ties;
    double tie_tol, recheck_tol;
    int32_t *recheck_list;      // FP32 pass: low-margin syndromes are appended here
    int32_t *recheck_count;
    int64_t recheck_cap;
};

// LDS written by some lanes of this wave is read by others: the LDS serves a
// wave's accesses in order, so only the compiler has to keep the order.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint32_t wave_field(uint32_t words, int i) {
    return (uint32_t)__builtin_amdgcn_readlane((int)words, i);
}

template <int CTRL>
__device__ __forceinline__ float wave_max_dpp(float x) {
    const float y = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, false));
    return y > x ? y : x;
}

// Maximum over the lanes that serve the same syndrome (equal low glog bits).
__device__ __forceinline__ float wave_max(float x, int glog) {
    const uint32_t u = __float_as_uint(x);
    const auto p32 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    x = fmaxf(__uint_as_float(p32[0]), __uint_as_float(p32[1]));
    const uint32_t v = __float_as_uint(x);
    const auto p16 = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    x = fmaxf(__uint_as_float(p16[0]), __uint_as_float(p16[1]));
    x = wave_max_dpp<0x128>(x);                      // row_ror:8
    if (glog < 3) x = wave_max_dpp<0x124>(x);        // row_ror:4
    if (glog < 2) x = wave_max_dpp<0x4E>(x);         // quad_perm [2,3,0,1]
    if (glog < 1) x = wave_max_dpp<0xB1>(x);         // quad_perm [1,0,3,2]
    return x;
}

// What one step's loops need: operand and output addresses of this lane
// before the output index's upper bits are known, strides in entries.
template <typename T>
struct WaveStep {
    const T *pa, *pb;
    T *pc;
    uint32_t idx;       // a's index | b's index << 16
    uint32_t c;         // output index
    int ka, kb;         // stride of a contracted term
    int nkk;            // contracted terms
    int hi, nhi;        // first and number of the output bits above the lane's
    int glog, shift;
};

// All outputs of a step, 2^UL at a time, KC contracted terms in flight.
template <typename T, bool SCALE, int KC, int UL>
__device__ __forceinline__ T wave_outputs(const WaveStep<T> &s, uint32_t words) {
    constexpr int U = 1 << UL;
    uint32_t dx[U], dc[U];
    dx[0] = dc[0] = 0;
#pragma unroll
    for (int u = 1; u < U; ++u) {
        const int bit = 31 - __builtin_clz(u);
        dx[u] = dx[u - (1 << bit)] ^ wave_field(words, kWaveBits + s.hi + bit);
        dc[u] = dc[u - (1 << bit)] | 1u << (s.hi + bit);
    }
    const int outer = 1 << (s.nhi - UL);
    uint32_t idx = s.idx, c = s.c;
    T lmax = 0;
    for (int o = 1;; ++o) {
        const T *pa[U], *pb[U];
        T acc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t x = idx ^ dx[u];
            pa[u] = s.pa + ((x & 0xffffu) << s.glog);
            pb[u] = s.pb + ((x >> 16) << s.glog);
            acc[u] = 0;
        }
        for (int k = 0; k < s.nkk; k += KC) {
            T va[KC][U], vb[KC][U];
#pragma unroll
            for (int j = 0; j < KC; ++j)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    va[j][u] = pa[u][(k + j) * s.ka];
                    vb[j][u] = pb[u][(k + j) * s.kb];
                }
#pragma unroll
            for (int j = 0; j < KC; ++j)
#pragma unroll
                for (int u = 0; u < U; ++u) acc[u] = fma(va[j][u], vb[j][u], acc[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (SCALE) {
                acc[u] = ldexp(acc[u], s.shift);
                lmax = acc[u] > lmax ? acc[u] : lmax;
            } else if (s.shift != 0) {
                acc[u] = ldexp(acc[u], s.shift);
            }
            s.pc[(c | dc[u]) << s.glog] = acc[u];
        }
        if (o >= outer) break;
        const int bit = s.hi + UL + __builtin_ctz(o);
        idx ^= wave_field(words, kWaveBits + bit);
        c ^= 1u << bit;
    }
    return lmax;
}

// The same for a step with labels summed on one side only, a term at a time.
template <typename T, bool SCALE>
__device__ __forceinline__ T wave_outputs_single(const WaveStep<T> &s, uint32_t words, int na, int sa, int nb, int sb) {
    const int outer = 1 << s.nhi;
    uint32_t idx = s.idx, c = s.c;
    T lmax = 0;
    for (int o = 1;; ++o) {
        const T *pa = s.pa + ((idx & 0xffffu) << s.glog), *pb = s.pb + ((idx >> 16) << s.glog);
        T acc = 0;
        for (int k = 0; k < s.nkk; ++k) {
            T va = 0, vb = 0;
            if (na == 1) va = pa[k * s.ka];
            else
                for (int q = 0; q < na; ++q) va += pa[k * s.ka + q * sa];
            if (nb == 1) vb = pb[k * s.kb];
            else
                for (int q = 0; q < nb; ++q) vb += pb[k * s.kb + q * sb];
            acc = fma(va, vb, acc);
        }
        if (SCALE) {
            acc = ldexp(acc, s.shift);
            lmax = acc > lmax ? acc : lmax;
        } else if (s.shift != 0) {
            acc = ldexp(acc, s.shift);
        }
        s.pc[c << s.glog] = acc;
        if (o >= outer) break;
        const int bit = s.hi + __builtin_ctz(o);
        idx ^= wave_field(words, kWaveBits + bit);
        c ^= 1u << bit;
    }
    return lmax;
}

template <typename T, bool SCALE, int KC>
__device__ __forceinline__ T wave_outputs_any(const WaveStep<T> &s, uint32_t words) {
    if (s.nhi >= 2) return wave_outputs<T, SCALE, KC, 2>(s, words);
    if (s.nhi == 1) return wave_outputs<T, SCALE, KC, 1>(s, words);
    return wave_outputs<T, SCALE, KC, 0>(s, words);
}

// Workgroups of any number of waves; waves stride over the tiles of
// G syndromes.  Dynamic LDS: d.desc_bytes(), then d.wave_bytes() per wave:
// values [ws + nent][G], scales mx/ex [nslots][G], slice bases [nops][G],
// syndrome bits [nbits + 1][G].
template <typename T, bool SCALE>
__global__ void __launch_bounds__(256) wave_kernel(WaveArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const int glog = a.d.glog, G = 1 << glog, g = lane & (G - 1), lc = lane >> glog, cl = 6 - glog;
    const T *tab = reinterpret_cast<const T *>(a.tab);
    const int64_t count = a.list ? (int64_t)(*a.list_count) : a.n;
    const int64_t ntiles = (count + G - 1) >> glog;
    if ((int64_t)blockIdx.x * waves >= ntiles) return;
    uint32_t *desc = reinterpret_cast<uint32_t *>(smem);
    const uint32_t *ops = desc + a.d.nsteps * kWaveWords;
    {
        const uint4 *src = reinterpret_cast<const uint4 *>(a.desc);
        uint4 *dst = reinterpret_cast<uint4 *>(smem);
        for (int i = tid; i < a.d.desc_bytes() / 16; i += blockDim.x) dst[i] = src[i];
    }
    unsigned char *mine = smem + a.d.desc_bytes() + wave * a.d.wave_bytes((int)sizeof(T));
    T *val = reinterpret_cast<T *>(mine);
    float *mx = reinterpret_cast<float *>(val + (a.d.vals() << glog));
    int *ex = reinterpret_cast<int *>(mx + (a.d.nslots << glog));
    uint32_t *base = reinterpret_cast<uint32_t *>(ex + (a.d.nslots << glog));
    uint8_t *bits = reinterpret_cast<uint8_t *>(base + (a.d.nops << glog));
    int lanebit[6];
#pragma unroll
    for (int t = 0; t < 6; ++t) lanebit[t] = t < cl ? -((lc >> t) & 1) : 0;
    __syncthreads();
    for (int64_t t = (int64_t)blockIdx.x * waves + wave; t < ntiles; t += (int64_t)gridDim.x * waves) {
        const int64_t qi = (t << glog) + g;
        const bool valid = qi < count;
        const int64_t qc = valid ? qi : count - 1;   // lanes beyond the last row read it again and store nothing
        const int64_t b = a.list ? (int64_t)a.list[qc] : qc;
        {
            const uint8_t *row = a.syn + b * a.d.nbits;
            for (int i = lc; i < a.d.nbits; i += 64 >> glog) bits[(i << glog) + g] = row[i] & 1u;
            bits[(a.d.nbits << glog) + g] = 0;
        }
        wave_lds_fence();
        // the slice that each staged operand takes
        for (int i = lc; i < a.d.nops; i += 64 >> glog) {
            const uint4 q = *reinterpret_cast<const uint4 *>(ops + i * kWaveOpWords);
            const uint2 r = *reinterpret_cast<const uint2 *>(ops + i * kWaveOpWords + 4);
            const uint32_t ev[4] = {q.z, q.w, r.x, r.y};
            uint32_t v = 0;
#pragma unroll
            for (int j = 0; j < kMaxEv; ++j)
                v |= (uint32_t)bits[(((ev[j >> 1] >> (16 * (j & 1))) & 0xffffu) << glog) + g] << j;
            base[(i << glog) + g] = q.x + (v << q.y);
        }
        wave_lds_fence();
        {
            T *dst = val + (a.d.ws << glog);
            const int n = a.d.nent << glog;
            for (int i = lane; i < n; i += 64 * 8) {
                T x[8];
                int at[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    at[u] = min(i + 64 * u, n - G + g);
                    const uint32_t e = a.ent[at[u] >> glog];
                    x[u] = tab[base[((e >> 16) << glog) + g] + (e & 0xffffu)];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) dst[at[u]] = x[u];
            }
        }
        wave_lds_fence();
        bool low = false;
        uint32_t next = lane < kWaveWords ? desc[lane] : 0u;
        for (int s = 0; s < a.d.nsteps; ++s) {
            const uint32_t words = next;
            next = lane < kWaveWords ? desc[min(s + 1, a.d.nsteps - 1) * kWaveWords + lane] : 0u;
            const uint32_t w0 = wave_field(words, 0), w4 = wave_field(words, 4);
            const bool aw = (w0 >> 16) & 1, bw = (w0 >> 17) & 1;
            WaveStep<T> st;
            st.glog = glog;
            int e = 0;
            if (SCALE) {
                int na = 0, nb = 0, ea, eb;
                if (aw) {
                    const int sl = (int)(wave_field(words, 6) << glog) + g;
                    const float m = mx[sl];
                    na = (m > 0.f) ? ilogbf(m) : 0;
                    ea = ex[sl] + na;
                    low = low || na < -100;
                } else {
                    ea = (int)wave_field(words, 9);
                }
                if (bw) {
                    const int sl = (int)(wave_field(words, 7) << glog) + g;
                    const float m = mx[sl];
                    nb = (m > 0.f) ? ilogbf(m) : 0;
                    eb = ex[sl] + nb;
                    low = low || nb < -100;
                } else {
                    eb = (int)wave_field(words, 10);
                }
                st.shift = -(na + nb);
                e = ea + eb;
            } else {
                st.shift = (int)wave_field(words, 9) + (int)wave_field(words, 10);
            }
            st.pa = val + (wave_field(words, 1) << glog) + g;
            st.pb = val + (wave_field(words, 2) << glog) + g;
            st.pc = val + (wave_field(words, 3) << glog) + g;
            st.idx = 0;
#pragma unroll
            for (int i = 0; i < 6; ++i) st.idx |= (uint32_t)lanebit[i] & wave_field(words, kWaveBits + i);
            const int rc = (int)(w0 & 0xffu), nk = (int)((w0 >> 8) & 0xffu);
            // lanes beyond a short output repeat the others' entries
            st.c = (uint32_t)lc & ((1u << rc) - 1u);
            st.hi = cl;
            st.nhi = max(0, rc - cl);
            st.nkk = 1 << nk;
            st.ka = 1 << ((int)(w4 & 0xffu) + glog);
            st.kb = 1 << ((int)((w4 >> 8) & 0xffu) + glog);
            T lmax;
            if ((w4 >> 16) != 0) {
                const uint32_t w5 = wave_field(words, 5);
                lmax = wave_outputs_single<T, SCALE>(st, words, 1 << ((w4 >> 16) & 0xffu), 1 << ((w5 & 0xffu) + glog),
                                                     1 << (w4 >> 24), 1 << (((w5 >> 8) & 0xffu) + glog));
            } else if (nk >= 2) {
                lmax = wave_outputs_any<T, SCALE, 4>(st, words);
            } else if (nk == 1) {
                lmax = wave_outputs_any<T, SCALE, 2>(st, words);
            } else {
                lmax = wave_outputs_any<T, SCALE, 1>(st, words);
            }
            if (SCALE) {
                const int sl = (int)(wave_field(words, 8) << glog) + g;
                mx[sl] = wave_max((float)lmax, glog);
                ex[sl] = e;
            }
            wave_lds_fence();
        }
        const T *root = val + (a.root_off << glog) + g;
        const int e = SCALE ? ex[(a.root_slot << glog) + g] : 0;
        if (valid && a.marginals)
            for (int j = lc; j < a.nout; j += 64 >> glog) a.marginals[b * a.nout + j] = ldexp((double)root[j << glog], e);
        if (valid && lane < G) {
            T best = 0, second = -1;
            int bi = 0;
            for (int j = 0; j < a.nout; ++j) {
                const T x = root[j << glog];
                if (j == 0 || x > best) {
                    if (j > 0) second = best;
                    best = x;
                    bi = j;
                } else if (x > second) {
                    second = x;
                }
            }
            if (a.classes) a.classes[b] = bi;
            const double gap = (double)(best - second);
            if (a.ties) a.ties[b] = (a.nout > 1 && second >= 0 && gap <= a.tie_tol * (double)best) ? 1 : 0;
            if (SCALE && a.recheck_list) {
                const bool rc = !(best > 0) || low || (a.nout > 1 && second >= 0 && gap <= a.recheck_tol * (double)best);
                if (rc) {
                    const int32_t slot = atomicAdd(a.recheck_count, 1);
                    if (slot < a.recheck_cap) a.recheck_list[slot] = (int32_t)b;
                }
            }
        }
        wave_lds_fence();
    }
}

}  // namespace tqec
