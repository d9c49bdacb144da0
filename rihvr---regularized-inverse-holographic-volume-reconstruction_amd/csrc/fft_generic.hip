// fft_generic.hip -- FFTs of run-time length (multiples of 16 up to 4096) for the forward operator
// A, its adjoint and the hologram transforms, where the compile-time plans of fft_kernels.hip do
// not cover the hologram size (the reference plans any size with cufftPlan2d(H, W),
// sparse_compressive_holo.cu:98).
//
// The same row and column passes as fft_kernels.hip (the same prologues and epilogues, the line
// occupancy and strip maps), with a plan chosen at run time: Stockham autosort passes (the indexing
// of fft.hpp) of radices 16, 8, 4, 2, 3, 5, 7, 9, 11, 13 in registers, and a direct DFT of any larger
// prime.  A workgroup holds several rows, or a strip of 16 columns (8 or 4 where 16 do not fit in
// LDS), in one LDS buffer: a pass reads its butterflies into registers, waits, and writes them
// back in place, so a transform moves its data through memory once.  (Before, columns ran as rows
// between tiled transposes, three passes over the volume for each of A and A^T, with the row passes
// limited by a division per butterfly and two LDS buffers.)
#include <algorithm>
#include <type_traits>

#include "fft.hpp"
#include "kernels.hpp"

namespace rihvr {

namespace {

constexpr int kGenMaxL = 4096;
constexpr int kGenMaxPasses = 12;
constexpr int kRowPer = 8;           // elements per thread of a row workgroup at most
constexpr int kRowMaxThreads = 512;
constexpr int kColLds = 160 * 1024;  // LDS of a column workgroup at most
constexpr int kColPer = 20;          // elements per thread of a column workgroup at most

// A pass of radix R after passes of total size Ns: nbf = L / R butterflies, twiddle step L / (Ns R);
// m_ns, m_nbf: 2^32 / d rounded up, for divisions by d (exact while the dividend times d is below
// 2^32: both are at most 4096)
struct GenPass {
    int R, Ns, nbf, step;
    unsigned m_ns, m_nbf;
    unsigned m_pair, m_out;  // radices above 13: for nbf h and nbf (h + 1), h = (R - 1) / 2
};
struct GenPlan {
    int L, np;
    unsigned m_l;  // for divisions by L
    GenPass p[kGenMaxPasses];
};

unsigned magic(int d) { return d > 1 ? (unsigned)(((1ull << 32) + d - 1) / d) : 0u; }
__device__ __forceinline__ int div_by(int x, int d, unsigned m) { return d > 1 ? (int)__umulhi((unsigned)x, m) : x; }

// Radices of L: its power of two (at least 16) in as few passes of radix up to max_radix (16, 8 or
// 4) as possible, evenly sized, the largest first (16 = 4 4: a plan has at least two passes); then
// 9s, then its other odd prime factors.  A second power of two goes last.
bool make_plan(int L, GenPlan* plan, int max_radix) {
    if (L < 16 || L > kGenMaxL || L % 16) return false;
    int bits = 0, odd = L;
    while (odd % 2 == 0) {
        odd /= 2;
        ++bits;
    }
    const int most = max_radix >= 16 && L > 16 ? 4 : max_radix >= 8 ? 3 : 2;
    const int n2 = (bits + most - 1) / most;
    int rad[kGenMaxPasses], n = 0, last = 0;
    for (int i = 0; i < n2; ++i) {
        const int b = (bits + n2 - 1 - i) / n2;
        if (i > 0 && i == n2 - 1) last = 1 << b;
        else rad[n++] = 1 << b;
    }
    while (odd % 9 == 0) {
        rad[n++] = 9;
        odd /= 9;
    }
    for (int f = 3; odd > 1; f += 2)
        while (odd % f == 0) {
            rad[n++] = f;
            odd /= f;
        }
    if (last) rad[n++] = last;
    plan->L = L;
    plan->np = n;
    plan->m_l = magic(L);
    int Ns = 1;
    for (int i = 0; i < n; ++i) {
        GenPass& p = plan->p[i];
        p.R = rad[i];
        p.Ns = Ns;
        p.nbf = L / p.R;
        p.step = L / (Ns * p.R);
        p.m_ns = magic(Ns);
        p.m_nbf = magic(p.nbf);
        p.m_pair = magic(p.nbf * ((p.R - 1) / 2));
        p.m_out = magic(p.nbf * ((p.R - 1) / 2 + 1));
        Ns *= p.R;
    }
    return true;
}

// Rows of length L that a row workgroup holds, and its threads (kRowPer elements each): the row
// count up to kRowMaxThreads whose last wave is fullest.  Row kernels take 8 elements per thread
// and radices up to 8: with 16 they need 200 to 256 VGPRs, one or two waves per SIMD.
int row_threads(int L, int rows) { return (rows * L / kRowPer + 63) / 64 * 64; }
int gen_rows_per_block(int L) {
    int best = 1;
    for (int r = 2; row_threads(L, r) <= kRowMaxThreads; ++r)
        if ((long)r * row_threads(L, best) >= (long)best * row_threads(L, r)) best = r;
    return best;
}

// How a workgroup's work items map to its transforms.  Items of a pass with n butterflies: (which
// transform, butterfly); at(which, j): LDS slot of element j.
struct RowMap {
    int tid, threads;
    int rows, lp;  // rows of the workgroup, LDS row pitch (element j at j + j / 16)
    static constexpr int kPer = kRowPer;
    __device__ __forceinline__ int stride() const { return threads; }
    __device__ __forceinline__ void split(int g, int n, unsigned m, int* which, int* b) const {
        *which = div_by(g, n, m);
        *b = g - *which * n;
    }
    __device__ __forceinline__ bool ok(int which, int, int) const { return which < rows; }
    __device__ __forceinline__ int slot(int which, int j) const { return which * lp + j + (j >> 4); }
};
struct ColMap {
    int tid, sh, threads;  // 2^sh columns
    static constexpr int kPer = kColPer;
    __device__ __forceinline__ int stride() const { return threads; }
    __device__ __forceinline__ void split(int g, int, unsigned, int* which, int* b) const {
        *which = g & ((1 << sh) - 1);
        *b = g >> sh;
    }
    __device__ __forceinline__ bool ok(int, int b, int n) const { return b < n; }
    __device__ __forceinline__ int slot(int which, int j) const { return (j << sh) + which; }
};

// One pass of compile-time radix R.  FIRST: elements come from src(slot, which, j), the slot a
// compile-time index of the thread's elements; LAST: results go to
// dst(which, j, v).
template <int R, int SIGN, bool FIRST, bool LAST, class Map, class Src, class Dst>
__device__ __forceinline__ void gen_pass(const GenPass& p, const Map& map, float2* buf, const float2* tw, Src&& src,
                                         Dst&& dst) {
    constexpr int NB = (Map::kPer + R - 1) / R;
    float2 v[NB][R];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        int which, b;
        map.split(map.tid + i * map.stride(), p.nbf, p.m_nbf, &which, &b);
        if (map.ok(which, b, p.nbf)) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if constexpr (FIRST)
                    v[i][r] = src(i * R + r, which, b + r * p.nbf);
                else
                    v[i][r] = buf[map.slot(which, b + r * p.nbf)];
            }
        }
    }
    if constexpr (!FIRST) __syncthreads();  // every butterfly is read before one is written in place
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        int which, b;
        map.split(map.tid + i * map.stride(), p.nbf, p.m_nbf, &which, &b);
        if (map.ok(which, b, p.nbf)) {
            const int q = FIRST ? b : div_by(b, p.Ns, p.m_ns), k = FIRST ? 0 : b - q * p.Ns;
            if constexpr (!FIRST) {
                const int ks = k * p.step;
#pragma unroll
                for (int r = 1; r < R; ++r) v[i][r] = cmul(v[i][r], tw[r * ks]);
            }
            Dft<R, SIGN, R>::run(v[i], nullptr);
            const int base = q * p.Ns * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if constexpr (LAST)
                    dst(which, base + r * p.Ns, v[i][r]);
                else
                    buf[map.slot(which, base + r * p.Ns)] = v[i][r];
            }
        }
    }
    if constexpr (!LAST) __syncthreads();
}

// A pass of any odd radix R = 2 h + 1 (a prime above 13), as fft.hpp's odd radices: the twiddled
// inputs j and R - j become their sum and difference in place, then an item forms outputs kk and
// R - kk (kk = 0: output 0) from the h pairs, with W_R^m = W_L^{m nbf} from the table.
template <bool LAST, class Map, class Dst>
__device__ __forceinline__ void gen_pass_any(const GenPass& p, const Map& map, float2* buf, const float2* tw,
                                             Dst&& dst) {
    const int h = (p.R - 1) / 2;
    constexpr int NP = (Map::kPer + 1) / 2, NO = (Map::kPer * 9 + 16) / 17;  // h / R < 1/2, (h + 1) / R <= 9/17
    for (int i = 0; i < NP; ++i) {
        int which, e;
        map.split(map.tid + i * map.stride(), p.nbf * h, p.m_pair, &which, &e);
        if (map.ok(which, e, p.nbf * h)) {
            const int j = div_by(e, p.nbf, p.m_nbf) + 1, b = e - (j - 1) * p.nbf;
            const int k = b - div_by(b, p.Ns, p.m_ns) * p.Ns;
            float2& x = buf[map.slot(which, b + j * p.nbf)];
            float2& y = buf[map.slot(which, b + (p.R - j) * p.nbf)];
            const float2 xt = cmul(x, tw[j * k * p.step]), yt = cmul(y, tw[(p.R - j) * k * p.step]);
            x = cadd(xt, yt);
            y = csub(xt, yt);
        }
    }
    __syncthreads();
    float2 lo[NO], hi[NO];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
        int which, e;
        map.split(map.tid + i * map.stride(), p.nbf * (h + 1), p.m_out, &which, &e);
        if (map.ok(which, e, p.nbf * (h + 1))) {
            const int kk = div_by(e, p.nbf, p.m_nbf), b = e - kk * p.nbf;
            float2 s = buf[map.slot(which, b)], d = make_float2(0.0f, 0.0f);
            int m = 0;
            for (int j = 1; j <= h; ++j) {
                m += kk;
                m = m >= p.R ? m - p.R : m;
                const float2 w = tw[m * p.nbf];
                const float2 x = buf[map.slot(which, b + j * p.nbf)], y = buf[map.slot(which, b + (p.R - j) * p.nbf)];
                s = make_float2(fmaf(x.x, w.x, s.x), fmaf(x.y, w.x, s.y));
                d = make_float2(fmaf(y.x, w.y, d.x), fmaf(y.y, w.y, d.y));
            }
            lo[i] = make_float2(s.x - d.y, s.y + d.x);
            hi[i] = make_float2(s.x + d.y, s.y - d.x);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NO; ++i) {
        int which, e;
        map.split(map.tid + i * map.stride(), p.nbf * (h + 1), p.m_out, &which, &e);
        if (map.ok(which, e, p.nbf * (h + 1))) {
            const int kk = div_by(e, p.nbf, p.m_nbf), b = e - kk * p.nbf;
            const int q = div_by(b, p.Ns, p.m_ns), base = q * p.Ns * p.R + (b - q * p.Ns);
            if constexpr (LAST) {
                dst(which, base + kk * p.Ns, lo[i]);
                if (kk) dst(which, base + (p.R - kk) * p.Ns, hi[i]);
            } else {
                buf[map.slot(which, base + kk * p.Ns)] = lo[i];
                if (kk) buf[map.slot(which, base + (p.R - kk) * p.Ns)] = hi[i];
            }
        }
    }
    if constexpr (!LAST) __syncthreads();
}

template <int SIGN, class Map, class Src>
__device__ __forceinline__ void first_pass(const GenPass& f, const Map& map, float2* buf, const float2* tw, Src&& src) {
    auto none = [](int, int, float2) {};
    switch (f.R) {
        case 16:
            if constexpr (Map::kPer >= 16) gen_pass<16, SIGN, true, false>(f, map, buf, tw, src, none);
            break;
        case 8: gen_pass<8, SIGN, true, false>(f, map, buf, tw, src, none); break;
        default: gen_pass<4, SIGN, true, false>(f, map, buf, tw, src, none); break;
    }
}

// The plan's passes: elements from src(slot, which, j), or where `full` (uniform) from
// src_full, which need not test whether its element is present; results to dst(which, j, v), or
// where dst is an int left in buf (each at its slot).
template <int SIGN, class Map, class Src, class SrcFull, class Dst>
__device__ __forceinline__ void run_plan(const GenPlan& pl, const Map& map, float2* buf, const float2* tw, bool full,
                                         SrcFull&& src_full, Src&& src, Dst&& dst) {
    constexpr bool kToLds = std::is_same<std::decay_t<Dst>, int>::value;
    auto none = [](int, int, float2) {};
    auto nosrc = [](int, int, int) { return make_float2(0.0f, 0.0f); };
    if constexpr (std::is_same<std::decay_t<Src>, int>::value) {
        first_pass<SIGN>(pl.p[0], map, buf, tw, src_full);
    } else {
        if (full)
            first_pass<SIGN>(pl.p[0], map, buf, tw, src_full);
        else
            first_pass<SIGN>(pl.p[0], map, buf, tw, src);
    }
    for (int i = 1; i < pl.np - (kToLds ? 0 : 1); ++i) {
        const GenPass& p = pl.p[i];
        switch (p.R) {
            case 16:
                if constexpr (Map::kPer >= 16) gen_pass<16, SIGN, false, false>(p, map, buf, tw, nosrc, none);
                break;
            case 8: gen_pass<8, SIGN, false, false>(p, map, buf, tw, nosrc, none); break;
            case 4: gen_pass<4, SIGN, false, false>(p, map, buf, tw, nosrc, none); break;
            case 2:
                if constexpr (kToLds) gen_pass<2, SIGN, false, false>(p, map, buf, tw, nosrc, none);
                break;
            case 3: gen_pass<3, SIGN, false, false>(p, map, buf, tw, nosrc, none); break;
            case 5: gen_pass<5, SIGN, false, false>(p, map, buf, tw, nosrc, none); break;
            case 7: gen_pass<7, SIGN, false, false>(p, map, buf, tw, nosrc, none); break;
            case 9: gen_pass<9, SIGN, false, false>(p, map, buf, tw, nosrc, none); break;
            default:
                if constexpr (Map::kPer >= 16) {
                    if (p.R == 11) {
                        gen_pass<11, SIGN, false, false>(p, map, buf, tw, nosrc, none);
                        break;
                    }
                    if (p.R == 13) {
                        gen_pass<13, SIGN, false, false>(p, map, buf, tw, nosrc, none);
                        break;
                    }
                }
                gen_pass_any<false>(p, map, buf, tw, none);
                break;
        }
    }
    if constexpr (!kToLds) {
        const GenPass& p = pl.p[pl.np - 1];
        switch (p.R) {
            case 16:
                if constexpr (Map::kPer >= 16) gen_pass<16, SIGN, false, true>(p, map, buf, tw, nosrc, dst);
                break;
            case 8: gen_pass<8, SIGN, false, true>(p, map, buf, tw, nosrc, dst); break;
            case 4: gen_pass<4, SIGN, false, true>(p, map, buf, tw, nosrc, dst); break;
            case 2: gen_pass<2, SIGN, false, true>(p, map, buf, tw, nosrc, dst); break;
            case 3: gen_pass<3, SIGN, false, true>(p, map, buf, tw, nosrc, dst); break;
            case 5: gen_pass<5, SIGN, false, true>(p, map, buf, tw, nosrc, dst); break;
            case 7: gen_pass<7, SIGN, false, true>(p, map, buf, tw, nosrc, dst); break;
            case 9: gen_pass<9, SIGN, false, true>(p, map, buf, tw, nosrc, dst); break;
            default:
                if constexpr (Map::kPer >= 16) {
                    if (p.R == 11) {
                        gen_pass<11, SIGN, false, true>(p, map, buf, tw, nosrc, dst);
                        break;
                    }
                    if (p.R == 13) {
                        gen_pass<13, SIGN, false, true>(p, map, buf, tw, nosrc, dst);
                        break;
                    }
                }
                gen_pass_any<true>(p, map, buf, tw, dst);
                break;
        }
    }
}

// fn(slot, which, j) for every element that this thread's first pass reads, in its slot order
template <int R, class Map, class F>
__device__ __forceinline__ void first_slots_r(const GenPass& p, const Map& map, F&& fn) {
    constexpr int NB = (Map::kPer + R - 1) / R;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        int which, b;
        map.split(map.tid + i * map.stride(), p.nbf, p.m_nbf, &which, &b);
        if (map.ok(which, b, p.nbf)) {
#pragma unroll
            for (int r = 0; r < R; ++r) fn(i * R + r, which, b + r * p.nbf);
        }
    }
}
template <class Map, class F>
__device__ __forceinline__ void first_slots(const GenPass& p, const Map& map, F&& fn) {
    switch (p.R) {
        case 8: first_slots_r<8>(p, map, fn); break;
        default: first_slots_r<4>(p, map, fn); break;
    }
}

// ----------------------------------------------------------------------------
// Row kernels (fft_kernels.hip's k_rows)
// ----------------------------------------------------------------------------
enum GenRowMode { GR_PLAIN = 0, GR_ADJ = 1, GR_FWDACC = 2, GR_SUMPART = 3 };

struct GenRowArgs {
    GenPlan plan;
    int rows, threads;    // of a workgroup
    const float2* in;     // PLAIN: [rows][L]; FWDACC: [nz][nrows][L]; SUMPART: [nparts][nrows][L]
    float2* out;          // PLAIN/SUMPART: [rows][L]; ADJ: [nz][nrows][L]; FWDACC: [chunks][nrows][L]
    const float2* tw;     // W_L^m for the transform's sign
    int nrows;            // rows per plane (ADJ, FWDACC) or in total (PLAIN, SUMPART)
    const float2* rhat;   // ADJ: [nrows][L]
    bool stream_out;      // ADJ: the output is larger than the caches
    const double* kappa;  // ADJ, FWDACC: [nrows][L]
    const float* zlist;
    int nz, zchunk;
    float invN;
    int nparts;
    long part_stride;
    const uint8_t* smap;  // FWDACC: 16-column strips present ([nz][L/16]; 0 = read as zeros)
};

inline int row_pitch(int L) { return L + L / 16 + 1; }

template <int SIGN, int MODE>
__global__ void __launch_bounds__(kRowMaxThreads, 5) k_gen_rows(GenRowArgs a) {
    extern __shared__ float2 gen_lds[];
    const int L = a.plan.L;
    const int row0 = blockIdx.x * a.rows;
    RowMap map{(int)threadIdx.x, a.threads, min(a.rows, a.nrows - row0), L + L / 16 + 1};
    float2* buf = gen_lds;
    float2* tw = gen_lds + a.rows * map.lp;
    for (int m = threadIdx.x; m < L; m += a.threads) tw[m] = a.tw[m];
    __syncthreads();
    if constexpr (MODE == GR_PLAIN || MODE == GR_SUMPART) {
        const float2* src = a.in + (size_t)row0 * L;
        float2* dst = a.out + (size_t)row0 * L;
        run_plan<SIGN>(
            a.plan, map, buf, tw, true,
            [&](int, int w, int j) {
                const int o = w * L + j;
                float2 v = src[o];
                if constexpr (MODE == GR_SUMPART)
                    for (int p = 1; p < a.nparts; ++p) v = cadd(v, src[(size_t)p * a.part_stride + o]);
                return v;
            },
            0,
            [&](int w, int j, float2 v) { dst[w * L + j] = v; });
    } else if constexpr (MODE == GR_ADJ) {
        // H_z R-hat / N, then the inverse FFT along x, for a chunk of planes; R-hat and kappa of the
        // thread's elements stay in registers
        float2 rh[kRowPer];
        double kp[kRowPer];
        const float2* rhp = a.rhat + (size_t)row0 * L;
        const double* kpp = a.kappa + (size_t)row0 * L;
#pragma unroll
        for (int i = 0; i < kRowPer; ++i) {
            rh[i] = make_float2(0.0f, 0.0f);
            kp[i] = 0.0;
        }
        first_slots(a.plan.p[0], map, [&](int s, int w, int j) {
            rh[s] = rhp[w * L + j];
            kp[s] = kpp[w * L + j];
        });
        const int z0 = blockIdx.y * a.zchunk, z1 = min(a.nz, z0 + a.zchunk);
        for (int z = z0; z < z1; ++z) {
            fresh(map.tid);
            const double zz = (double)a.zlist[z];
            float2* dst = a.out + ((size_t)z * a.nrows + row0) * L;
            run_plan<SIGN>(
                a.plan, map, buf, tw, true,
                [&](int s, int, int) { return cscale(cmul(transfer(zz, kp[s]), rh[s]), a.invN); }, 0,
                [&](int w, int j, float2 v) { store_stream(dst + (w * L + j), v, a.stream_out); });
        }
    } else {  // GR_FWDACC: forward FFT along x, times H_{-z}, summed over a chunk of planes
        // the transform's results stay in LDS and are taken from there in raster order, so that a
        // thread's sums and kappa have the same few registers whatever the last radix
        float2 acc[kRowPer];
        double kp[kRowPer];
        const double* kpp = a.kappa + (size_t)row0 * L;
        const int n = map.rows * L;
#pragma unroll
        for (int i = 0; i < kRowPer; ++i) {
            const int o = threadIdx.x + i * a.threads;
            acc[i] = make_float2(0.0f, 0.0f);
            kp[i] = o < n ? kpp[o] : 0.0;
        }
        const int z0 = blockIdx.y * a.zchunk, z1 = min(a.nz, z0 + a.zchunk);
        const int NS = L / 16;  // strips per row, at most 256
        const int lane = threadIdx.x & 63;
        for (int z = z0; z < z1; ++z) {
            // the plane's strips as wave-uniform masks (every wave reads the same bytes); a plane
            // without any adds zeros, so it is skipped by the whole workgroup
            const uint8_t* sm = a.smap + (size_t)z * NS;
            uint64_t m[kGenMaxL / 1024];
            int present = 0;
#pragma unroll
            for (int k = 0; k < kGenMaxL / 1024; ++k) {
                const int s = k * 64 + lane;
                m[k] = k * 64 < NS ? __ballot(s < NS && sm[s < NS ? s : 0] != 0) : 0ull;
                present += __popcll(m[k]);
            }
            if (!present) continue;
            fresh(map.tid);
            const double mz = -(double)a.zlist[z];
            const float2* src = a.in + ((size_t)z * a.nrows + row0) * L;
            run_plan<SIGN>(
                a.plan, map, buf, tw, present == NS, [&](int, int w, int j) { return src[w * L + j]; },
                [&](int, int w, int j) {
                    const uint64_t mk = j < 1024 ? m[0] : j < 2048 ? m[1] : j < 3072 ? m[2] : m[3];
                    return ((mk >> ((j >> 4) & 63)) & 1ull) ? src[w * L + j] : make_float2(0.0f, 0.0f);
                },
                0);
#pragma unroll
            for (int i = 0; i < kRowPer; ++i) {
                const int o = threadIdx.x + i * a.threads;
                if (o < n) {
                    const int w = div_by(o, L, a.plan.m_l);
                    acc[i] = cadd(acc[i], cmul(transfer(mz, kp[i]), buf[map.slot(w, o - w * L)]));
                }
            }
            __syncthreads();
        }
        float2* dst = a.out + (size_t)blockIdx.y * a.part_stride + (size_t)row0 * L;
#pragma unroll
        for (int i = 0; i < kRowPer; ++i) {
            const int o = threadIdx.x + i * a.threads;
            if (o < n) dst[o] = acc[i];
        }
    }
}

template <int SIGN, int MODE> hipError_t launch_rows(GenRowArgs& a, int L, int radix, unsigned gy, hipStream_t s) {
    if (!make_plan(L, &a.plan, std::min(radix, 8))) return hipErrorInvalidValue;
    a.rows = gen_rows_per_block(L);
    a.threads = row_threads(L, a.rows);
    const unsigned gx = (unsigned)((a.nrows + a.rows - 1) / a.rows);
    if (gx == 0 || gy == 0) return hipSuccess;
    const size_t lds = ((size_t)a.rows * row_pitch(L) + L) * sizeof(float2);
    hipLaunchKernelGGL((k_gen_rows<SIGN, MODE>), dim3(gx, gy), dim3(a.threads), lds, s, a);
    return hipGetLastError();
}

// ----------------------------------------------------------------------------
// Column kernels (fft_kernels.hip's k_cols): a workgroup transforms 2^sh adjacent columns of one
// plane, 16 where they fit in LDS with the twiddle table.
// ----------------------------------------------------------------------------
enum GenColMode { GC_PLAIN = 0, GC_ADJ = 1, GC_FWD = 2, GC_REAL = 3 };

struct GenColArgs {
    GenPlan plan;
    int sh, threads;
    const float2* in;  // [planes][L][W]
    float2* out;
    int W, nstrips;    // strips of 2^sh columns per plane
    const float2* tw;
    const float2* phase;  // ADJ, FWD
    const float2* meas;   // REAL
    float2* resid;
    double* partial;
    const uint64_t* occ;         // FWD: line occupancy of the input (may be NULL), its plane words
    const uint64_t* occ_planes;  // (may be NULL) and the strip map written
    uint8_t* smap;
    int lsh;  // a line is 2^lsh columns
};

template <int SIGN, int MODE> __global__ void __launch_bounds__(1024) k_gen_cols(GenColArgs a) {
    extern __shared__ float2 gen_lds[];
    __shared__ double red_s[17];
    __shared__ uint32_t rows_s[kGenMaxL / 32];
    // neighbouring strips, which share memory lines where they are narrower than 16 columns, run
    // on one XCD
    const int lb = xcd_local_block(blockIdx.x, gridDim.x);
    const int z = lb / a.nstrips, strip = lb - z * a.nstrips;
    const int L = a.plan.L;
    const ColMap map{(int)threadIdx.x, a.sh, a.threads};
    float2* buf = gen_lds;
    float2* tw = gen_lds + ((size_t)L << a.sh);
    const int col0 = strip << a.sh;
    const size_t W = (size_t)a.W;
    const float2* src = a.in + (size_t)z * L * W + col0;
    if constexpr (MODE == GC_FWD) {
        // rows whose line is empty are not read; a strip without any transforms to zeros, which are
        // not written (the strip map tells the row pass).  The strips of a 16-column group lie in
        // one line, so they agree on the map's byte.
        const int line = col0 >> a.lsh;
        const bool plane_set = !a.occ_planes || ((a.occ_planes[z] >> line) & 1ull);
        uint8_t* sm = a.smap + (size_t)z * (W / 16) + (col0 >> 4);
        if (!plane_set) {
            if (threadIdx.x == 0) *sm = 0;
            return;
        }
        const uint64_t* occ = a.occ ? a.occ + (size_t)z * L : nullptr;
        for (int k = threadIdx.x; k < (L + 31) / 32; k += a.threads) rows_s[k] = occ ? 0u : ~0u;
        __syncthreads();
        bool mine = false;
        if (occ)
            for (int j = threadIdx.x; j < L; j += a.threads)
                if ((occ[j] >> line) & 1ull) {
                    atomicOr(&rows_s[j >> 5], 1u << (j & 31));
                    mine = true;
                }
        const bool any = occ ? __syncthreads_or(mine) : true;
        if (threadIdx.x == 0) *sm = any ? 1 : 0;
        if (!any) return;
    }
    for (int m = threadIdx.x; m < L; m += a.threads) tw[m] = a.tw[m];
    __syncthreads();
    if constexpr (MODE == GC_PLAIN || MODE == GC_ADJ) {
        float2* dst = a.out + (size_t)z * L * W + col0;
        float2 ph = make_float2(1.0f, 0.0f);
        if constexpr (MODE == GC_ADJ) ph = a.phase[z];
        const bool wide = a.sh >= 4;  // whole memory lines (narrower strips share them through the caches)
        run_plan<SIGN>(
            a.plan, map, buf, tw, true,
            [&](int, int w, int j) { return load_stream(src + ((size_t)j * W + w), MODE == GC_ADJ && wide); }, 0,
            [&](int w, int j, float2 v) {
                if constexpr (MODE == GC_ADJ) v = make_float2(v.x * ph.x - v.y * ph.y, v.y * ph.x + v.x * ph.y);
                store_stream(dst + ((size_t)j * W + w), v, MODE == GC_ADJ && wide);
            });
    } else if constexpr (MODE == GC_FWD) {
        const float2 ph = a.phase[z];
        const float px = ph.x, py = -ph.y;
        float2* dst = a.out + (size_t)z * L * W + col0;
        run_plan<SIGN>(
            a.plan, map, buf, tw, !a.occ,
            [&](int, int w, int j) {
                const float2 d = src[(size_t)j * W + w];
                return make_float2(d.x * px - d.y * py, d.y * px + d.x * py);
            },
            [&](int, int w, int j) {
                if (!((rows_s[j >> 5] >> (j & 31)) & 1u)) return make_float2(0.0f, 0.0f);
                const float2 d = src[(size_t)j * W + w];
                return make_float2(d.x * px - d.y * py, d.y * px + d.x * py);
            },
            [&](int w, int j, float2 v) { dst[(size_t)j * W + w] = v; });
    } else {  // GC_REAL: est = Re(IFFT(...)), r = est - meas, partial sum |r|^2
        double s = 0.0;
        run_plan<SIGN>(
            a.plan, map, buf, tw, true, [&](int, int w, int j) { return src[(size_t)j * W + w]; }, 0,
            [&](int w, int j, float2 v) {
                const size_t o = (size_t)j * W + col0 + w;
                const float2 e = make_float2(v.x, 0.0f);  // back_propagate_finish_kernel
                a.out[o] = e;
                const float2 m = a.meas[o];
                const float2 r = make_float2(e.x - m.x, e.y - m.y);  // RM_EST_TRUE
                a.resid[o] = r;
                s += (double)r.x * r.x + (double)r.y * r.y;
            });
        const double tot = block_sum(s, red_s);
        if (threadIdx.x == 0) a.partial[strip] = tot;
    }
}

// 2^sh columns per workgroup: the widest of 16, 8, 4, 2 whose strip and twiddle table fit in LDS
// beside the kernels' own arrays
int col_shift(int L) {
    const size_t room = kColLds - 1024;
    for (int sh = 4; sh > 1; --sh)
        if ((((size_t)L << sh) + L) * sizeof(float2) <= room && ((long)L << sh) <= 1024L * kColPer) return sh;
    return 1;
}

template <int SIGN, int MODE> hipError_t launch_cols(GenColArgs& a, int L, int radix, int nz, hipStream_t s) {
    if (!make_plan(L, &a.plan, radix) || a.W % 16) return hipErrorInvalidValue;
    a.sh = col_shift(L);
    a.nstrips = a.W >> a.sh;
    // 16 elements per thread, up to 1024 threads (then up to kColPer)
    a.threads = (int)std::min<long>(1024, ((((long)L << a.sh) + 15) / 16 + 63) / 64 * 64);
    const long blocks = (long)a.nstrips * nz;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    const size_t lds = (((size_t)L << a.sh) + L) * sizeof(float2);
    hipLaunchKernelGGL((k_gen_cols<SIGN, MODE>), dim3((unsigned)blocks), dim3(a.threads), lds, s, a);
    return hipGetLastError();
}

}  // namespace

bool gen_fft_supported(int L) {
    GenPlan p;
    return make_plan(L, &p, 16);
}

int gen_rows_blocks(int L, int H) { return (H + gen_rows_per_block(L) - 1) / gen_rows_per_block(L); }
int gen_cols_blocks(int L, int W) { return W >> col_shift(L); }

hipError_t gen_rows_plain(int L, int radix, int sign, const float2* in, float2* out, int nrows, const float2* tw,
                          hipStream_t s) {
    GenRowArgs a{};
    a.in = in; a.out = out; a.tw = tw; a.nrows = nrows;
    return sign < 0 ? launch_rows<-1, GR_PLAIN>(a, L, radix, 1, s) : launch_rows<1, GR_PLAIN>(a, L, radix, 1, s);
}

hipError_t gen_rows_sumparts(int L, int radix, const float2* parts, int nparts, long part_stride, float2* out,
                             int nrows, const float2* tw_inv, hipStream_t s) {
    GenRowArgs a{};
    a.in = parts; a.out = out; a.tw = tw_inv; a.nrows = nrows; a.nparts = nparts; a.part_stride = part_stride;
    return launch_rows<1, GR_SUMPART>(a, L, radix, 1, s);
}

hipError_t gen_rows_adj(int L, int radix, const float2* rhat, const double* kappa, const float* zlist, float2* out,
                        int nrows, int nz, int zchunk, float invN, const float2* tw_inv, hipStream_t s) {
    if (zchunk < 1) return hipErrorInvalidValue;
    GenRowArgs a{};
    a.out = out; a.tw = tw_inv; a.nrows = nrows; a.rhat = rhat; a.kappa = kappa; a.zlist = zlist; a.nz = nz;
    a.zchunk = zchunk; a.invN = invN;
    a.stream_out = streams(L, nrows, nz);
    return launch_rows<1, GR_ADJ>(a, L, radix, (unsigned)((nz + zchunk - 1) / zchunk), s);
}

hipError_t gen_rows_fwdacc(int L, int radix, const float2* in, const double* kappa, const float* zlist, float2* parts,
                           int nrows, int nz, int zchunk, const float2* tw_fwd, const uint8_t* smap, hipStream_t s) {
    if (zchunk < 1) return hipErrorInvalidValue;
    GenRowArgs a{};
    a.in = in; a.out = parts; a.tw = tw_fwd; a.nrows = nrows; a.kappa = kappa; a.zlist = zlist; a.nz = nz;
    a.zchunk = zchunk; a.part_stride = (long)nrows * L; a.smap = smap;
    return launch_rows<-1, GR_FWDACC>(a, L, radix, (unsigned)((nz + zchunk - 1) / zchunk), s);
}

hipError_t gen_cols_plain(int L, int radix, int sign, const float2* in, float2* out, int W, int nplanes,
                          const float2* tw, hipStream_t s) {
    GenColArgs a{};
    a.in = in; a.out = out; a.W = W; a.tw = tw;
    return sign < 0 ? launch_cols<-1, GC_PLAIN>(a, L, radix, nplanes, s) : launch_cols<1, GC_PLAIN>(a, L, radix, nplanes, s);
}

hipError_t gen_cols_adj(int L, int radix, const float2* in, const float2* phase, float2* out, int W, int nz,
                        const float2* tw_inv, hipStream_t s) {
    GenColArgs a{};
    a.in = in; a.out = out; a.W = W; a.tw = tw_inv; a.phase = phase;
    return launch_cols<1, GC_ADJ>(a, L, radix, nz, s);
}

hipError_t gen_cols_fwd(int L, int radix, const float2* in, const float2* phase, float2* out, int W, int nz,
                        const float2* tw_fwd, const uint64_t* occ, const uint64_t* occ_planes, uint8_t* smap,
                        hipStream_t s) {
    GenColArgs a{};
    a.in = in; a.out = out; a.W = W; a.tw = tw_fwd; a.phase = phase; a.occ = occ; a.occ_planes = occ_planes;
    a.smap = smap; a.lsh = line_shift(W);
    return launch_cols<-1, GC_FWD>(a, L, radix, nz, s);
}

hipError_t gen_cols_real(int L, int radix, const float2* in, float2* est, const float2* meas, float2* resid,
                         double* partial, int W, const float2* tw_inv, hipStream_t s) {
    GenColArgs a{};
    a.in = in; a.out = est; a.W = W; a.tw = tw_inv; a.meas = meas; a.resid = resid; a.partial = partial;
    return launch_cols<1, GC_REAL>(a, L, radix, 1, s);
}

}  // namespace rihvr
