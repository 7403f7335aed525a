// sampler_hip.hip — on-device syndrome sampling and error-pattern recovery.
//
// Sampler: replaces the reference's per-sample loop of
// `random_error_pattern(em)` (src/decoding/error_model.jl:69-71, 97-117)
// followed by `syndrome_extraction` (:131-146).  Draws come from
// Philox4x32-10 with counter (column j, sample mod 2^32, sample >> 32,
// stream tag) and key (seed mod 2^32, seed >> 32), converted to a double with
// 53 random bits, so every sample is bit-identical to the host sampler.
// A workgroup takes 64 samples bit by bit: a wave draws one variable for all
// 64 and the ballot of the lanes that flip is the variable's mask, and a
// syndrome or class bit of all 64 is the XOR of its members' masks.
//
// Recovery: replaces `error_pattern` (src/decoding/tndecoder.jl:167-174) and
// its MIP pure-error solve (src/decoding/ipdecoder.jl:150-169) by a GF(2)
// right inverse: e = R s, then the reference's logical fix per class bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "tqec_hip.h"

namespace tqec {
int set_error_shared(int code, const std::string &msg);  // tqec_hip.hip: backs tqec_last_error()
}

namespace {

int fail(int code, const std::string &m) { return tqec::set_error_shared(code, m); }

constexpr int kMaxSynWords = 8;   // up to 512 syndrome bits
constexpr int kMaxErrWords = 16;  // up to 1024 error variables per pattern half

__device__ __forceinline__ void philox10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c[0], p1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
        const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
        c[0] = n0;
        c[1] = (uint32_t)p1;
        c[2] = n2;
        c[3] = (uint32_t)p0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

__device__ __forceinline__ double uniform53(uint32_t x0, uint32_t x1) {
    const double a = (double)(x0 >> 5), b = (double)(x1 >> 6);
    return (a * 67108864.0 + b) * (1.0 / 9007199254740992.0);
}

// Rows of a binary matrix as lists of column numbers, on the device.
struct RowLists {
    int32_t *ptr = nullptr;   // [rows + 1]
    int32_t *idx = nullptr;
};

struct SamplerArgs {
    int kind;            // 0: CSS depolarizing, 1: independent flips
    int nvar;            // qubits (kind 0) or mechanisms (kind 1)
    int nsyn;            // syndrome bits
    int nlog;            // logical class bits
    int synw;            // 64-bit words per syndrome column
    const double *t1, *t2, *t3;   // kind 0: py, px+py, px+py+pz; kind 1: t1 = p
    // thresholds of the drawn 53-bit integers, [nvar][3]: u < t exactly when
    // the integer is below ceil(t 2^53)
    const unsigned long long *cut;
    // members of each syndrome bit, then of each class bit: 2 j for an X error
    // of qubit j and 2 j + 1 for a Z error (kind 0), j (kind 1)
    RowLists rows;
    // kind 0: per qubit, the syndrome column of an X error and of a Z error
    // and the logical-class column of each; kind 1: column of the mechanism
    const unsigned long long *colx, *colz;   // [nvar][synw]
    const uint32_t *logx, *logz;             // [nvar]
    uint32_t seed_lo, seed_hi, stream_tag;
    int64_t first, n;
    uint8_t *syn;        // [n][nsyn]
    int32_t *cls;        // [n] or null
    uint8_t *err;        // kind 0: [n][2 nvar] (x bits then z bits); kind 1: [n][nvar]; or null
    // the same as masks of 64 samples (bit i: sample 64 b + i), or null
    unsigned long long *synm;   // [ceil(n / 64)][nsyn]
    unsigned long long *errm;   // [ceil(n / 64)][2 nvar] (2 j: x, 2 j + 1: z) or [..][nvar]
};

// Bit i of a mask, by its 32-bit half.  Two builds of the max-product wave
// kernel took such bits with a 64-bit shift by a vector register, and in some
// runs a few rows came out with one wrong bit (always of the same label, the
// log-probabilities right); the same source with 32-bit halves gave none in 60
// configurations of 60 runs.  Reading the two builds showed no missing wait or
// ordering between lanes, so the cause is not known, and no kernel of the
// library shifts 64 bits by a vector register any more (shifts by a scalar
// register, as of a uniform index, were never seen to fail).
__device__ __forceinline__ uint32_t mask_bit(unsigned long long m, int i) {
    const uint32_t w = i < 32 ? (uint32_t)m : (uint32_t)(m >> 32);
    return (w >> (i & 31)) & 1u;
}

// Rows of `width` bytes of samples [0, rows) out to `out`, byte c of a sample
// being its bit of mask at(c).  Four bytes per store where `out` allows it.
template <typename At>
__device__ __forceinline__ void store_bits(uint8_t *__restrict__ out, int rows, int width, const At &at) {
    const int total = rows * width, t0 = threadIdx.x, nt = blockDim.x;
    int done = 0;
    if (((uintptr_t)out & 3) == 0) {
        done = total & ~3;
        for (int f = 4 * t0; f < done; f += 4 * nt) {
            int i = f / width, c = f - i * width;
            uint32_t v = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v |= mask_bit(at(c), i) << (8 * e);
                if (++c == width) {
                    c = 0;
                    ++i;
                }
            }
            *reinterpret_cast<uint32_t *>(out + f) = v;
        }
    }
    for (int f = done + t0; f < total; f += nt) {
        const int i = f / width;
        out[f] = (uint8_t)mask_bit(at(f - i * width), i);
    }
}

__device__ __forceinline__ unsigned long long xor_list(const RowLists &m, int row, const unsigned long long *mask) {
    unsigned long long x = 0ull;
    const int end = m.ptr[row + 1];
#pragma unroll 4
    for (int e = m.ptr[row]; e < end; ++e) x ^= mask[m.idx[e]];
    return x;
}

// Bound by the Philox multiplies (17 of 64 bits per draw: with the variable
// uniform over the wave, the first round and half of the second are scalar or
// outside the loop).  Measured at 49 qubits, 65,536 samples: 12 us with masks
// of the errors, against 71 us for a thread per sample that stored every error
// bit as a byte of its own row.  LDS: the masks of all variables, syndrome and
// class bits.
__global__ void __launch_bounds__(256) sample_kernel(SamplerArgs a) {
    extern __shared__ unsigned long long masks[];
    const int es = a.kind == 0 ? 2 : 1;
    unsigned long long *err = masks, *row = masks + (size_t)es * a.nvar;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t b0 = (int64_t)blockIdx.x * 64;
    const int rows = (int)min((int64_t)64, a.n - b0);
    const unsigned long long s = (unsigned long long)(a.first + b0 + lane);
    const uint32_t s_lo = (uint32_t)s, s_hi = (uint32_t)(s >> 32);
    for (int j = wave; j < a.nvar; j += 4) {
        uint32_t c[4] = {(uint32_t)j, s_lo, s_hi, a.stream_tag};
        philox10(c, a.seed_lo, a.seed_hi);
        const unsigned long long u = ((unsigned long long)(c[0] >> 5) << 26) | (c[1] >> 6);
        const unsigned long long *cut = a.cut + 3 * j;
        if (a.kind == 0) {
            const bool y = u < cut[0];
            const bool x = !y && u < cut[1];
            const bool z = !y && !x && u < cut[2];
            const unsigned long long mx = __ballot(y || x), mz = __ballot(y || z);
            if (lane < 2) err[2 * j + lane] = lane ? mz : mx;
        } else {
            const unsigned long long m = __ballot(u < cut[0]);
            if (lane == 0) err[j] = m;
        }
    }
    __syncthreads();
    for (int r = threadIdx.x; r < a.nsyn + a.nlog; r += 256) row[r] = xor_list(a.rows, r, err);
    if (a.errm)
        for (int t = threadIdx.x; t < es * a.nvar; t += 256) a.errm[(int64_t)blockIdx.x * es * a.nvar + t] = err[t];
    __syncthreads();
    if (a.synm)
        for (int t = threadIdx.x; t < a.nsyn; t += 256) a.synm[(int64_t)blockIdx.x * a.nsyn + t] = row[t];
    store_bits(a.syn + b0 * a.nsyn, rows, a.nsyn, [&](int c) { return row[c]; });
    if (a.cls && (int)threadIdx.x < rows) {
        uint32_t c = 0;
        for (int l = 0; l < a.nlog; ++l) c |= mask_bit(row[a.nsyn + l], threadIdx.x) << l;
        a.cls[b0 + threadIdx.x] = (int32_t)c;
    }
    if (a.err) {
        const int nv = a.nvar;
        if (a.kind == 0)
            store_bits(a.err + b0 * 2 * nv, rows, 2 * nv, [&](int c) { return err[c < nv ? 2 * c : 2 * (c - nv) + 1]; });
        else
            store_bits(a.err + b0 * nv, rows, nv, [&](int c) { return err[c]; });
    }
}

// LDS that the masks may take; models with more variables use the kernel below.
constexpr size_t kSampleLds = 60 * 1024;

size_t sample_lds(int es, int nvar, int nsyn, int nlog) { return ((size_t)es * nvar + nsyn + nlog) * 8; }

// One thread per sample, for models whose masks outgrow the LDS (above 3,700
// qubits or 7,500 mechanisms).
__global__ void sample_large_kernel(SamplerArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const int64_t s = a.first + i;
    unsigned long long acc[kMaxSynWords];
    for (int w = 0; w < kMaxSynWords; ++w) acc[w] = 0ull;
    uint32_t lg = 0;
    for (int j = 0; j < a.nvar; ++j) {
        uint32_t c[4] = {(uint32_t)j, (uint32_t)(s & 0xffffffffll), (uint32_t)((unsigned long long)s >> 32),
                         a.stream_tag};
        philox10(c, a.seed_lo, a.seed_hi);
        const double u = uniform53(c[0], c[1]);
        bool fx, fz;
        if (a.kind == 0) {
            const bool y = u < a.t1[j];
            const bool x = !y && u < a.t2[j];
            const bool z = !y && !x && u < a.t3[j];
            fx = y || x;
            fz = y || z;
        } else {
            fx = u < a.t1[j];
            fz = false;
        }
        if (fx) {
            for (int w = 0; w < a.synw; ++w) acc[w] ^= a.colx[(int64_t)j * a.synw + w];
            lg ^= a.logx[j];
        }
        if (fz) {
            for (int w = 0; w < a.synw; ++w) acc[w] ^= a.colz[(int64_t)j * a.synw + w];
            lg ^= a.logz[j];
        }
        if (a.err) {
            if (a.kind == 0) {
                a.err[i * 2 * a.nvar + j] = fx;
                a.err[i * 2 * a.nvar + a.nvar + j] = fz;
            } else {
                a.err[i * a.nvar + j] = fx;
            }
        }
    }
    uint8_t *row = a.syn + i * a.nsyn;
    for (int b = 0; b < a.nsyn; ++b) row[b] = (uint8_t)((acc[b >> 6] >> (b & 63)) & 1ull);
    if (a.cls) a.cls[i] = (int32_t)lg;
}

struct RecoveryArgs {
    int nq;              // error variables per half
    int nsa, nsb;        // syndrome bits feeding half a (ex <- sz) and half b (ez <- sx)
    int ew;              // 64-bit words per error pattern half
    int k;               // logical pairs (CSS) or logicals (DEM)
    int kind;            // 0: CSS; 1: DEM with the reference's logical fix
    int nsyn;            // bytes per syndrome row
    int offa, offb;      // first syndrome bit of each half's syndrome
    const unsigned long long *Ra, *Rb;   // [nsa][ew], [nsb][ew]: columns of the right inverses
    const unsigned long long *la, *lb;   // [k][ew]: CSS: lz (test ex), lx (test ez); DEM: l2q masks
    const unsigned long long *fa, *fb;   // [k][ew]: CSS: lx (added to ex), lz (added to ez)
    const uint8_t *syn;
    const int32_t *cls;
    int64_t n;
    uint8_t *ea, *eb;    // [n][nq] each (eb unused for DEM)
};

__global__ void recovery_kernel(RecoveryArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const uint8_t *row = a.syn + i * a.nsyn;
    unsigned long long ea[kMaxErrWords], eb[kMaxErrWords];
    for (int w = 0; w < kMaxErrWords; ++w) ea[w] = eb[w] = 0ull;
    for (int j = 0; j < a.nsa; ++j)
        if (row[a.offa + j] & 1)
            for (int w = 0; w < a.ew; ++w) ea[w] ^= a.Ra[(int64_t)j * a.ew + w];
    for (int j = 0; j < a.nsb; ++j)
        if (row[a.offb + j] & 1)
            for (int w = 0; w < a.ew; ++w) eb[w] ^= a.Rb[(int64_t)j * a.ew + w];
    const int32_t c = a.cls[i];
    for (int l = 0; l < a.k; ++l) {
        if (a.kind == 0) {
            // tndecoder.jl:170: lz_l . ex must equal class bit k+l, else ex += lx_l
            int par = 0;
            for (int w = 0; w < a.ew; ++w) par ^= __popcll(ea[w] & a.la[l * a.ew + w]) & 1;
            if (par != ((c >> (a.k + l)) & 1))
                for (int w = 0; w < a.ew; ++w) ea[w] ^= a.fa[l * a.ew + w];
            // tndecoder.jl:171: lx_l . ez must equal class bit l, else ez += lz_l
            par = 0;
            for (int w = 0; w < a.ew; ++w) par ^= __popcll(eb[w] & a.lb[l * a.ew + w]) & 1;
            if (par != ((c >> l) & 1))
                for (int w = 0; w < a.ew; ++w) eb[w] ^= a.fb[l * a.ew + w];
        } else {
            // tndecoder.jl:263-269: when the parity of the mechanisms touching
            // logical l disagrees with the class, every one of them is flipped
            int par = 0;
            for (int w = 0; w < a.ew; ++w) par ^= __popcll(ea[w] & a.la[l * a.ew + w]) & 1;
            if (par != ((c >> l) & 1))
                for (int w = 0; w < a.ew; ++w) ea[w] ^= a.la[l * a.ew + w];
        }
    }
    for (int q = 0; q < a.nq; ++q) a.ea[i * a.nq + q] = (uint8_t)((ea[q >> 6] >> (q & 63)) & 1ull);
    if (a.kind == 0 && a.eb)
        for (int q = 0; q < a.nq; ++q) a.eb[i * a.nq + q] = (uint8_t)((eb[q >> 6] >> (q & 63)) & 1ull);
}

// Recovery and logical-error check of 64 samples per workgroup, on masks of
// the samples as the sampler leaves them: the recovered pattern (as
// recovery_kernel: right inverse, then the logical fix), its difference d from
// the sampled one, d's logical class bits (`check_logical_error`,
// src/decoding/error_model.jl:161-181, of every logical row at once) and d's
// syndrome, which must be zero when the recovered pattern reproduces the
// sampled syndrome.  counts: [0] samples with a logical error, [1] with one in
// the X-error half (lz . dx odd for some row; DEM: 0), [2] in the Z-error half
// (lx . dz odd), [3] recovered patterns that do not reproduce the syndrome.
// Measured at 49 qubits, 65,536 samples: 7 us, against 68 us for a recovery
// and a check that passed one byte per qubit through memory.
struct CheckArgs {
    int kind, nvar, nsyn, nlog, k;
    RowLists syn;              // members of each syndrome and class bit (the sampler's)
    RowLists inv;              // per error variable (2 j: x, 2 j + 1: z, or j): the syndrome bits its right inverse adds up
    RowLists test, add;        // per half and logical (half * k + l): variables whose parity is tested / flipped
    const unsigned long long *synm, *errm;
    const int32_t *cls;
    int64_t n;
    unsigned long long *counts;
};

__global__ void __launch_bounds__(256) ler_check_kernel(CheckArgs a) {
    extern __shared__ unsigned long long masks[];
    const int es = a.kind == 0 ? 2 : 1, nm = es * a.nvar;
    unsigned long long *syn = masks, *want = syn + a.nsyn, *pat = want + a.nlog, *out = pat + nm;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t b0 = (int64_t)blockIdx.x * 64;
    const int rows = (int)min((int64_t)64, a.n - b0);
    for (int r = tid; r < a.nsyn; r += 256) syn[r] = a.synm[(int64_t)blockIdx.x * a.nsyn + r];
    if (wave == 0) {
        const int32_t c = lane < rows ? a.cls[b0 + lane] : 0;
        for (int l = 0; l < a.nlog; ++l) {
            const unsigned long long m = __ballot((c >> l) & 1);
            if (lane == 0) want[l] = m;
        }
    }
    if (tid < 4) out[tid] = 0ull;
    __syncthreads();
    for (int v = tid; v < nm; v += 256) pat[v] = xor_list(a.inv, v, syn);
    __syncthreads();
    // tndecoder.jl:170-171 / :263-269: one wave per half, a logical after the other
    if (wave < es)
        for (int l = 0; l < a.k; ++l) {
            const int row = wave * a.k + l;
            unsigned long long par = 0ull;
            for (int e = a.test.ptr[row] + lane; e < a.test.ptr[row + 1]; e += 64) par ^= pat[a.test.idx[e]];
            for (int o = 32; o > 0; o >>= 1) par ^= __shfl_xor(par, o);
            // class bit k + l decides the X half (wave 0) of a CSS code, bit l the Z half
            const unsigned long long flip = par ^ want[a.kind == 0 && wave == 0 ? a.k + l : l];
            for (int e = a.add.ptr[row] + lane; e < a.add.ptr[row + 1]; e += 64) pat[a.add.idx[e]] ^= flip;
            // the next logical reads what other lanes have written here
            __threadfence_block();
            __builtin_amdgcn_wave_barrier();
        }
    __syncthreads();
    for (int v = tid; v < nm; v += 256) pat[v] ^= a.errm[(int64_t)blockIdx.x * nm + v];
    __syncthreads();
    for (int r = tid; r < a.nsyn + a.nlog; r += 256) {
        const unsigned long long x = xor_list(a.syn, r, pat);
        if (!x) continue;
        if (r < a.nsyn) {
            atomicOr(&out[3], x);
        } else {
            atomicOr(&out[0], x);
            if (a.kind == 0) atomicOr(&out[r - a.nsyn < a.k ? 2 : 1], x);
        }
    }
    __syncthreads();
    if (tid < 4) {
        const unsigned long long m = out[tid] & (rows == 64 ? ~0ull : (1ull << rows) - 1ull);
        if (m) atomicAdd(&a.counts[tid], (unsigned long long)__popcll(m));
    }
}

__global__ void ler_zero_kernel(unsigned long long *c) {
    if (threadIdx.x < 4) c[threadIdx.x] = 0ull;
}

#define TQS_HIP(call)                                                                      \
    do {                                                                                   \
        hipError_t e_ = (call);                                                            \
        if (e_ != hipSuccess) return fail(TQEC_EDEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <typename T>
int upload(const std::vector<T> &h, T **d) {
    TQS_HIP(hipMalloc((void **)d, std::max<size_t>(1, h.size()) * sizeof(T)));
    if (!h.empty()) TQS_HIP(hipMemcpy(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    return TQEC_OK;
}

std::vector<unsigned long long> pack_rows(const uint8_t *M, int rows, int cols, int words) {
    // M is rows x cols (row-major); returns [rows][words] bit-packed rows
    std::vector<unsigned long long> out((size_t)rows * words, 0ull);
    for (int r = 0; r < rows; ++r)
        for (int c = 0; c < cols; ++c)
            if (M[(size_t)r * cols + c] & 1) out[(size_t)r * words + (c >> 6)] |= 1ull << (c & 63);
    return out;
}

}  // namespace

namespace {

// Lists of the set columns of each row (rows given one after the other).
struct RowBuilder {
    std::vector<int32_t> ptr{0}, idx;
    void end_row() { ptr.push_back((int32_t)idx.size()); }
    int upload_to(RowLists *out) {
        int rc;
        if ((rc = upload(ptr, &out->ptr))) return rc;
        return upload(idx, &out->idx);
    }
};

void free_rows(RowLists &m) {
    (void)hipFree(m.ptr);
    (void)hipFree(m.idx);
}

// ceil(t 2^53) of the thresholds of each variable, three per variable.
std::vector<unsigned long long> cuts(const std::vector<double> &t1, const std::vector<double> &t2,
                                     const std::vector<double> &t3) {
    std::vector<unsigned long long> c;
    for (size_t j = 0; j < t1.size(); ++j)
        for (const std::vector<double> *t : {&t1, &t2, &t3})
            c.push_back(t->empty() ? 0ull : (unsigned long long)std::ceil(std::ldexp((*t)[j], 53)));
    return c;
}

}  // namespace

struct tqec_sampler {
    int kind = 0, nvar = 0, nsyn = 0, nlog = 0, synw = 0;
    uint32_t stream_tag = 0;
    double *t1 = nullptr, *t2 = nullptr, *t3 = nullptr;
    unsigned long long *colx = nullptr, *colz = nullptr;
    uint32_t *logx = nullptr, *logz = nullptr;
    unsigned long long *cut = nullptr;
    RowLists rows;
};

struct tqec_recovery {
    RecoveryArgs a{};
    RowLists inv, test, add;   // see CheckArgs
    unsigned long long *Ra = nullptr, *Rb = nullptr, *la = nullptr, *lb = nullptr, *fa = nullptr, *fb = nullptr;
};

struct tqec_ler {
    tqec_plan *plan = nullptr;
    tqec_sampler *smp = nullptr;
    tqec_recovery *rec = nullptr;
    int64_t batch = 0;
    uint8_t *syn = nullptr;
    int32_t *cls = nullptr;
    unsigned long long *synm = nullptr, *errm = nullptr;   // masks of 64 samples
    unsigned long long *counts = nullptr;
};

namespace {

SamplerArgs sampler_args(const tqec_sampler *s, uint64_t seed, int64_t first, int64_t n) {
    SamplerArgs a{};
    a.kind = s->kind;
    a.nvar = s->nvar;
    a.nsyn = s->nsyn;
    a.nlog = s->nlog;
    a.synw = s->synw;
    a.t1 = s->t1;
    a.t2 = s->t2;
    a.t3 = s->t3;
    a.colx = s->colx;
    a.colz = s->colz;
    a.logx = s->logx;
    a.logz = s->logz;
    a.seed_lo = (uint32_t)(seed & 0xffffffffull);
    a.seed_hi = (uint32_t)(seed >> 32);
    a.stream_tag = s->stream_tag;
    a.first = first;
    a.n = n;
    a.cut = s->cut;
    a.rows = s->rows;
    return a;
}

// Samples of one launch: a grid holds fewer than 2^32 work-items, and the
// kernel below takes four per sample.
constexpr int64_t kSampleLaunch = int64_t(1) << 29;

int launch_sample(const SamplerArgs &all, hipStream_t stream) {
    const int es = all.kind == 0 ? 2 : 1;
    const size_t lds = sample_lds(es, all.nvar, all.nsyn, all.nlog);
    for (int64_t off = 0; off < all.n; off += kSampleLaunch) {
        SamplerArgs a = all;
        a.first += off;
        a.n = std::min(kSampleLaunch, all.n - off);
        a.syn += off * a.nsyn;
        if (a.cls) a.cls += off;
        if (a.err) a.err += off * es * a.nvar;
        if (a.synm) a.synm += off / 64 * a.nsyn;
        if (a.errm) a.errm += off / 64 * es * a.nvar;
        if (lds <= kSampleLds)
            hipLaunchKernelGGL(sample_kernel, dim3((unsigned)((a.n + 63) / 64)), dim3(256), lds, stream, a);
        else
            hipLaunchKernelGGL(sample_large_kernel, dim3((unsigned)((a.n + 255) / 256)), dim3(256), 0, stream, a);
        TQS_HIP(hipGetLastError());
    }
    return TQEC_OK;
}

}  // namespace

extern "C" {

int tqec_sampler_create_css(int32_t nq, const double *px, const double *py, const double *pz, int32_t nsx,
                            const uint8_t *Hx, int32_t nsz, const uint8_t *Hz, int32_t k, const uint8_t *lx,
                            const uint8_t *lz, tqec_sampler **out) {
    if (!out || !px || !py || !pz || (nsx && !Hx) || (nsz && !Hz) || (k && (!lx || !lz)))
        return fail(TQEC_ENULL, "null argument");
    *out = nullptr;
    const int ns = nsx + nsz;
    if (nq <= 0 || ns <= 0 || ns > 64 * kMaxSynWords || k < 0 || 2 * k > 31)
        return fail(TQEC_EUNSUPPORTED, "sampler sizes out of range");
    for (int j = 0; j < nq; ++j)
        if (!(px[j] >= 0 && py[j] >= 0 && pz[j] >= 0 && px[j] + py[j] + pz[j] <= 1))
            return fail(TQEC_EINVAL, "probabilities must be non-negative with px+py+pz <= 1");
    auto *s = new (std::nothrow) tqec_sampler();
    if (!s) return fail(TQEC_ENOMEM, "out of host memory");
    s->kind = 0;
    s->nvar = nq;
    s->nsyn = ns;
    s->nlog = 2 * k;
    s->synw = (ns + 63) / 64;
    s->stream_tag = 0x51D0;
    std::vector<double> t1(nq), t2(nq), t3(nq);
    for (int j = 0; j < nq; ++j) {
        t1[j] = py[j];
        t2[j] = px[j] + py[j];
        t3[j] = px[j] + py[j] + pz[j];
    }
    // An X error on qubit j flips the Z checks holding j (sz = Hz ex) and the
    // class bit k+i when lz_i holds j; a Z error flips X checks and bit i.
    std::vector<unsigned long long> cx((size_t)nq * s->synw, 0), cz((size_t)nq * s->synw, 0);
    std::vector<uint32_t> lgx(nq, 0), lgz(nq, 0);
    for (int j = 0; j < nq; ++j) {
        for (int r = 0; r < nsx; ++r)
            if (Hx[(size_t)r * nq + j] & 1) cz[(size_t)j * s->synw + (r >> 6)] |= 1ull << (r & 63);
        for (int r = 0; r < nsz; ++r) {
            const int b = nsx + r;
            if (Hz[(size_t)r * nq + j] & 1) cx[(size_t)j * s->synw + (b >> 6)] |= 1ull << (b & 63);
        }
        for (int i = 0; i < k; ++i) {
            if (lz[(size_t)i * nq + j] & 1) lgx[j] |= 1u << (k + i);
            if (lx[(size_t)i * nq + j] & 1) lgz[j] |= 1u << i;
        }
    }
    RowBuilder rb;
    for (int r = 0; r < ns; ++r, rb.end_row())
        for (int j = 0; j < nq; ++j)
            if ((r < nsx ? Hx[(size_t)r * nq + j] : Hz[(size_t)(r - nsx) * nq + j]) & 1)
                rb.idx.push_back(2 * j + (r < nsx ? 1 : 0));
    for (int l = 0; l < 2 * k; ++l, rb.end_row())
        for (int j = 0; j < nq; ++j)
            if ((l < k ? lx[(size_t)l * nq + j] : lz[(size_t)(l - k) * nq + j]) & 1)
                rb.idx.push_back(2 * j + (l < k ? 1 : 0));
    int rc;
    if ((rc = upload(cuts(t1, t2, t3), &s->cut)) || (rc = rb.upload_to(&s->rows)) ||
        (rc = upload(t1, &s->t1)) || (rc = upload(t2, &s->t2)) || (rc = upload(t3, &s->t3)) ||
        (rc = upload(cx, &s->colx)) || (rc = upload(cz, &s->colz)) || (rc = upload(lgx, &s->logx)) ||
        (rc = upload(lgz, &s->logz))) {
        tqec_sampler_destroy(s);
        return rc;
    }
    *out = s;
    return TQEC_OK;
}

int tqec_sampler_create_flips(int32_t nm, const double *p, int32_t nd, const uint8_t *D, int32_t nl,
                              const uint8_t *Lm, tqec_sampler **out) {
    if (!out || !p || (nd && !D) || (nl && !Lm)) return fail(TQEC_ENULL, "null argument");
    *out = nullptr;
    if (nm <= 0 || nd <= 0 || nd > 64 * kMaxSynWords || nl < 0 || nl > 31)
        return fail(TQEC_EUNSUPPORTED, "sampler sizes out of range");
    for (int j = 0; j < nm; ++j)
        if (!(p[j] >= 0 && p[j] <= 1)) return fail(TQEC_EINVAL, "probabilities must be in [0, 1]");
    auto *s = new (std::nothrow) tqec_sampler();
    if (!s) return fail(TQEC_ENOMEM, "out of host memory");
    s->kind = 1;
    s->nvar = nm;
    s->nsyn = nd;
    s->nlog = nl;
    s->synw = (nd + 63) / 64;
    s->stream_tag = 0xF11B;
    std::vector<double> t1(p, p + nm);
    std::vector<unsigned long long> cx((size_t)nm * s->synw, 0);
    std::vector<uint32_t> lg(nm, 0);
    for (int j = 0; j < nm; ++j) {
        for (int r = 0; r < nd; ++r)
            if (D[(size_t)r * nm + j] & 1) cx[(size_t)j * s->synw + (r >> 6)] |= 1ull << (r & 63);
        for (int l = 0; l < nl; ++l)
            if (Lm[(size_t)l * nm + j] & 1) lg[j] |= 1u << l;
    }
    RowBuilder rb;
    for (int r = 0; r < nd + nl; ++r, rb.end_row())
        for (int j = 0; j < nm; ++j)
            if ((r < nd ? D[(size_t)r * nm + j] : Lm[(size_t)(r - nd) * nm + j]) & 1) rb.idx.push_back(j);
    int rc;
    if ((rc = upload(cuts(t1, {}, {}), &s->cut)) || (rc = rb.upload_to(&s->rows)) || (rc = upload(t1, &s->t1)) ||
        (rc = upload(cx, &s->colx)) || (rc = upload(lg, &s->logx))) {
        tqec_sampler_destroy(s);
        return rc;
    }
    *out = s;
    return TQEC_OK;
}

int tqec_sample(tqec_sampler *s, uint64_t seed, int64_t first, int64_t n, uint8_t *d_syndromes,
                int32_t *d_classes, uint8_t *d_errors, void *stream) {
    if (!s || (n > 0 && !d_syndromes)) return fail(TQEC_ENULL, "null argument");
    if (n < 0 || first < 0) return fail(TQEC_EINVAL, "negative count or offset");
    if (n == 0) return TQEC_OK;
    SamplerArgs a = sampler_args(s, seed, first, n);
    a.syn = d_syndromes;
    a.cls = d_classes;
    a.err = d_errors;
    return launch_sample(a, (hipStream_t)stream);
}

void tqec_sampler_destroy(tqec_sampler *s) {
    if (!s) return;
    (void)hipFree(s->t1);
    (void)hipFree(s->t2);
    (void)hipFree(s->t3);
    (void)hipFree(s->colx);
    (void)hipFree(s->colz);
    (void)hipFree(s->logx);
    (void)hipFree(s->logz);
    (void)hipFree(s->cut);
    free_rows(s->rows);
    delete s;
}

int tqec_recovery_create_css(int32_t nq, int32_t nsx, int32_t nsz, const uint8_t *Rx, const uint8_t *Rz,
                             int32_t k, const uint8_t *lx, const uint8_t *lz, tqec_recovery **out) {
    if (!out || !Rx || !Rz || (k && (!lx || !lz))) return fail(TQEC_ENULL, "null argument");
    *out = nullptr;
    if (nq <= 0 || nq > 64 * kMaxErrWords || nsx < 0 || nsz < 0 || k < 0 || 2 * k > 31)
        return fail(TQEC_EUNSUPPORTED, "recovery sizes out of range");
    auto *r = new (std::nothrow) tqec_recovery();
    if (!r) return fail(TQEC_ENOMEM, "out of host memory");
    const int ew = (nq + 63) / 64;
    // Rx: nq x nsz maps sz -> ex; columns packed as [nsz][ew]
    std::vector<uint8_t> tx((size_t)nsz * nq), tz((size_t)nsx * nq);
    for (int q = 0; q < nq; ++q) {
        for (int j = 0; j < nsz; ++j) tx[(size_t)j * nq + q] = Rx[(size_t)q * nsz + j];
        for (int j = 0; j < nsx; ++j) tz[(size_t)j * nq + q] = Rz[(size_t)q * nsx + j];
    }
    RowBuilder inv, test, add;
    for (int q = 0; q < nq; ++q)
        for (int half = 0; half < 2; ++half, inv.end_row())
            for (int j = 0; j < (half ? nsx : nsz); ++j)
                if ((half ? Rz[(size_t)q * nsx + j] : Rx[(size_t)q * nsz + j]) & 1) inv.idx.push_back(half ? j : nsx + j);
    for (int half = 0; half < 2; ++half)
        for (int l = 0; l < k; ++l, test.end_row(), add.end_row())
            for (int q = 0; q < nq; ++q) {
                if ((half ? lx : lz)[(size_t)l * nq + q] & 1) test.idx.push_back(2 * q + half);
                if ((half ? lz : lx)[(size_t)l * nq + q] & 1) add.idx.push_back(2 * q + half);
            }
    int rc;
    if ((rc = inv.upload_to(&r->inv)) || (rc = test.upload_to(&r->test)) || (rc = add.upload_to(&r->add)) ||
        (rc = upload(pack_rows(tx.data(), nsz, nq, ew), &r->Ra)) ||
        (rc = upload(pack_rows(tz.data(), nsx, nq, ew), &r->Rb)) ||
        (rc = upload(pack_rows(lz, k, nq, ew), &r->la)) || (rc = upload(pack_rows(lx, k, nq, ew), &r->lb)) ||
        (rc = upload(pack_rows(lx, k, nq, ew), &r->fa)) || (rc = upload(pack_rows(lz, k, nq, ew), &r->fb))) {
        tqec_recovery_destroy(r);
        return rc;
    }
    RecoveryArgs &a = r->a;
    a.nq = nq;
    a.nsa = nsz;
    a.nsb = nsx;
    a.ew = ew;
    a.k = k;
    a.kind = 0;
    a.nsyn = nsx + nsz;
    a.offa = nsx;
    a.offb = 0;
    a.Ra = r->Ra;
    a.Rb = r->Rb;
    a.la = r->la;
    a.lb = r->lb;
    a.fa = r->fa;
    a.fb = r->fb;
    *out = r;
    return TQEC_OK;
}

int tqec_recovery_create_dem(int32_t nm, int32_t nd, const uint8_t *R, int32_t nl, const uint8_t *l2q,
                             tqec_recovery **out) {
    if (!out || !R || (nl && !l2q)) return fail(TQEC_ENULL, "null argument");
    *out = nullptr;
    if (nm <= 0 || nm > 64 * kMaxErrWords || nd <= 0 || nl < 0 || nl > 31)
        return fail(TQEC_EUNSUPPORTED, "recovery sizes out of range");
    auto *r = new (std::nothrow) tqec_recovery();
    if (!r) return fail(TQEC_ENOMEM, "out of host memory");
    const int ew = (nm + 63) / 64;
    std::vector<uint8_t> t((size_t)nd * nm);
    for (int q = 0; q < nm; ++q)
        for (int j = 0; j < nd; ++j) t[(size_t)j * nm + q] = R[(size_t)q * nd + j];
    RowBuilder inv, test, add;
    for (int q = 0; q < nm; ++q, inv.end_row())
        for (int j = 0; j < nd; ++j)
            if (R[(size_t)q * nd + j] & 1) inv.idx.push_back(j);
    for (int l = 0; l < nl; ++l, test.end_row(), add.end_row())
        for (int q = 0; q < nm; ++q)
            if (l2q[(size_t)l * nm + q] & 1) {
                test.idx.push_back(q);
                add.idx.push_back(q);
            }
    int rc;
    if ((rc = inv.upload_to(&r->inv)) || (rc = test.upload_to(&r->test)) || (rc = add.upload_to(&r->add)) ||
        (rc = upload(pack_rows(t.data(), nd, nm, ew), &r->Ra)) || (rc = upload(pack_rows(l2q, nl, nm, ew), &r->la))) {
        tqec_recovery_destroy(r);
        return rc;
    }
    RecoveryArgs &a = r->a;
    a.nq = nm;
    a.nsa = nd;
    a.nsb = 0;
    a.ew = ew;
    a.k = nl;
    a.kind = 1;
    a.nsyn = nd;
    a.offa = 0;
    a.Ra = r->Ra;
    a.la = r->la;
    *out = r;
    return TQEC_OK;
}

int tqec_recover(tqec_recovery *r, const uint8_t *d_syndromes, const int32_t *d_classes, int64_t n,
                 uint8_t *d_err_a, uint8_t *d_err_b, void *stream) {
    if (!r || (n > 0 && (!d_syndromes || !d_classes || !d_err_a))) return fail(TQEC_ENULL, "null argument");
    if (n < 0) return fail(TQEC_EINVAL, "negative count");
    if (n == 0) return TQEC_OK;
    RecoveryArgs a = r->a;
    a.syn = d_syndromes;
    a.cls = d_classes;
    a.n = n;
    a.ea = d_err_a;
    a.eb = d_err_b;
    hipLaunchKernelGGL(recovery_kernel, dim3((unsigned)((n + 127) / 128)), dim3(128), 0, (hipStream_t)stream, a);
    TQS_HIP(hipGetLastError());
    return TQEC_OK;
}

int tqec_ler_create(tqec_plan *plan, tqec_sampler *smp, tqec_recovery *rec, int64_t batch, tqec_ler **out) {
    if (!out || !plan || !smp || !rec) return fail(TQEC_ENULL, "null argument");
    *out = nullptr;
    if (batch <= 0 || batch > (int64_t(1) << 24)) return fail(TQEC_EINVAL, "batch must be in [1, 2^24]");
    tqec_stats st{};
    int rc;
    if ((rc = tqec_plan_stats(plan, &st))) return rc;
    const RecoveryArgs &ra = rec->a;
    if (ra.kind != smp->kind || ra.nq != smp->nvar || ra.nsyn != smp->nsyn)
        return fail(TQEC_EINVAL, "sampler and recovery describe different codes");
    if (ra.kind == 0 ? (2 * ra.k != smp->nlog) : (ra.k != smp->nlog))
        return fail(TQEC_EINVAL, "sampler and recovery have different logical counts");
    if (st.n_out != smp->nlog) return fail(TQEC_EINVAL, "plan and sampler have different logical counts");
    auto *h = new (std::nothrow) tqec_ler();
    if (!h) return fail(TQEC_ENOMEM, "out of host memory");
    h->plan = plan;
    h->smp = smp;
    h->rec = rec;
    h->batch = batch;
    const size_t B = (size_t)batch, nv = (size_t)smp->nvar;
    const size_t blocks = (B + 63) / 64;
    hipError_t e = hipMalloc((void **)&h->syn, B * smp->nsyn);
    if (e == hipSuccess) e = hipMalloc((void **)&h->cls, B * sizeof(int32_t));
    if (e == hipSuccess) e = hipMalloc((void **)&h->synm, blocks * smp->nsyn * 8);
    if (e == hipSuccess) e = hipMalloc((void **)&h->errm, blocks * nv * (smp->kind == 0 ? 2 : 1) * 8);
    if (e == hipSuccess) e = hipMalloc((void **)&h->counts, 4 * sizeof(unsigned long long));
    if (e != hipSuccess) {
        tqec_ler_destroy(h);
        return fail(TQEC_ENOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    }
    *out = h;
    return TQEC_OK;
}

int tqec_ler_run(tqec_ler *h, int32_t mode, uint64_t seed, int64_t first, int64_t n, int64_t *counts, void *stream) {
    if (!h || !counts) return fail(TQEC_ENULL, "null argument");
    if (n < 0 || first < 0) return fail(TQEC_EINVAL, "negative count or offset");
    const hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(ler_zero_kernel, dim3(1), dim3(64), 0, st, h->counts);
    TQS_HIP(hipGetLastError());
    int rc;
    for (int64_t off = 0; off < n; off += h->batch) {
        const int64_t nb = std::min(h->batch, n - off);
        SamplerArgs sa = sampler_args(h->smp, seed, first + off, nb);
        sa.syn = h->syn;
        sa.synm = h->synm;
        sa.errm = h->errm;
        if ((rc = launch_sample(sa, st))) return rc;
        if ((rc = tqec_decode_batch_device(h->plan, h->syn, nb, mode, nullptr, h->cls, nullptr, stream))) return rc;
        CheckArgs a{};
        a.kind = h->smp->kind;
        a.nvar = h->smp->nvar;
        a.nsyn = h->smp->nsyn;
        a.nlog = h->smp->nlog;
        a.k = h->rec->a.k;
        a.syn = h->smp->rows;
        a.inv = h->rec->inv;
        a.test = h->rec->test;
        a.add = h->rec->add;
        a.synm = h->synm;
        a.errm = h->errm;
        a.cls = h->cls;
        a.n = nb;
        a.counts = h->counts;
        hipLaunchKernelGGL(ler_check_kernel, dim3((unsigned)((nb + 63) / 64)), dim3(256),
                           sample_lds(a.kind == 0 ? 2 : 1, a.nvar, a.nsyn, a.nlog + 4), st, a);
        TQS_HIP(hipGetLastError());
    }
    unsigned long long c[4];
    TQS_HIP(hipMemcpyAsync(c, h->counts, sizeof(c), hipMemcpyDeviceToHost, st));
    TQS_HIP(hipStreamSynchronize(st));
    for (int i = 0; i < 4; ++i) counts[i] = (int64_t)c[i];
    return TQEC_OK;
}

void tqec_ler_destroy(tqec_ler *h) {
    if (!h) return;
    (void)hipFree(h->syn);
    (void)hipFree(h->cls);
    (void)hipFree(h->synm);
    (void)hipFree(h->errm);
    (void)hipFree(h->counts);
    delete h;
}

void tqec_recovery_destroy(tqec_recovery *r) {
    if (!r) return;
    (void)hipFree(r->Ra);
    (void)hipFree(r->Rb);
    (void)hipFree(r->la);
    (void)hipFree(r->lb);
    (void)hipFree(r->fa);
    (void)hipFree(r->fb);
    free_rows(r->inv);
    free_rows(r->test);
    free_rows(r->add);
    delete r;
}

}  // extern "C"
