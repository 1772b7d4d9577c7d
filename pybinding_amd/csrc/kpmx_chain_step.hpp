// The chained diagonal recurrence: several Chebyshev steps per launch, written for gfx950 (MI355X).
//
// A single step reads r_k (gathered) and r_{k-1} and writes r_{k+1}: three passes over the vector
// block per step for a few multiply-adds per element, so a large block is bound by HBM bytes and a
// small one by the launch and the chain index load -> gather -> store inside it.  Here a workgroup
// takes a tile of consecutive rows together with the rows within distance K of it (its halo), holds
// r_k of all of them in LDS and r_{k-1} in registers, and runs K steps there: step j computes the
// rows within distance K - j, so after K steps the tile's own rows are exact and nothing is read
// from another workgroup.  A launch reads two vectors (halo rows twice) and writes two: 4 / K
// passes per step, and one launch for K steps.  The halo's redundant work is what limits K: the
// plan (build_chain in kpmx_abi.hip) weighs both from the tiles' measured halo sizes.
//
// Measured, single steps before and chained steps now, in us per step (K the steps per launch):
//   fp64, 32 vectors, 1.05 M sites, one hopping   155    65   K = 6, 96 us per launch of 8 columns
//   fp32, 32 vectors, 1.2 M sites, one hopping     93    50   K = 5, of 16 columns
//   fp64, 1 vector, 2.1 M sites                    26   5.8   K = 5
//   fp64, 24 vectors, 123 k rows of 19 entries     88    29   K = 3, of 8 columns
//   complex128, 16 vectors, 512 k sites            69    51   K = 5, of 4 columns, stored values
//   fp64, 8 vectors, 61 k sites                   5.8   2.0   K = 8
//   fp32, 1 vector, 137 k sites                   4.7   1.4   K = 12
// Large blocks are bound by their passes over memory (load and store phases take about half of a
// launch) beside LDS gathers and arithmetic, small ones by the latency of a step: two barriers, the
// gather and the sums.  Narrower column groups hold taller tiles but measured slower (fp64 block of 32:
// 8.4, 9.6 and 10.9 ms in groups of 8, 4 and 2; complex128 of 16: 6.6 and 8.7 ms in groups of 4 and 2;
// fp32 of 32: 6.8, 7.8 and 8.1 ms in groups of 16, 8 and 4).
//
// Layout: an item is one element of up to 16 bytes (a column pair, four fp32 columns, ...) of one
// local row; item i sits at X[i] and belongs to thread i % T for the whole launch, so r_{k-1} needs
// no LDS (half the footprint: tiles of twice the rows, or two workgroups per CU).  A step gathers
// from X and keeps r_{k+1} in registers, a barrier, then swaps it with X; a second barrier opens
// the next step.  Matrix entries are 2-byte local columns.
#pragma once
#include "kpmx_chain.hpp"
#include "kpmx_device.hpp"

#include <atomic>
#include <type_traits>
#include <utility>

namespace kpmx {
namespace {

// ------------------------------------------------------------------------------ elements
struct fquad {
    float v[4];
};
struct cpair {
    cf32 v[2];
};

template <class E> struct elem;
template <> struct elem<float>  { using value = float;  using real = float;  static constexpr int cols = 1, kinds = 2; };
template <> struct elem<double> { using value = double; using real = double; static constexpr int cols = 1, kinds = 2; };
template <> struct elem<dpair>  { using value = double; using real = double; static constexpr int cols = 2, kinds = 2; };
template <> struct elem<fquad>  { using value = float;  using real = float;  static constexpr int cols = 4, kinds = 2; };
template <> struct elem<cf32>   { using value = cf32;   using real = float;  static constexpr int cols = 1, kinds = 3; };
template <> struct elem<cpair>  { using value = cf32;   using real = float;  static constexpr int cols = 2, kinds = 3; };
template <> struct elem<cf64>   { using value = cf64;   using real = double; static constexpr int cols = 1, kinds = 3; };

template <class E> __device__ __forceinline__ E make_zero() { return zero(E{}); }
template <> __device__ __forceinline__ fquad make_zero<fquad>() { return {{0.f, 0.f, 0.f, 0.f}}; }
template <> __device__ __forceinline__ cpair make_zero<cpair>() { return {{{0.f, 0.f}, {0.f, 0.f}}}; }

__device__ __forceinline__ fquad fmac(float a, fquad b, fquad c) {
    return {{a * b.v[0] + c.v[0], a * b.v[1] + c.v[1], a * b.v[2] + c.v[2], a * b.v[3] + c.v[3]}};
}
__device__ __forceinline__ cpair fmac(cf32 a, cpair b, cpair c) {
    return {{kpmx::fmac(a, b.v[0], c.v[0]), kpmx::fmac(a, b.v[1], c.v[1])}};
}
__device__ __forceinline__ fquad scal(fquad a, float s) {
    return {{a.v[0] * s, a.v[1] * s, a.v[2] * s, a.v[3] * s}};
}
__device__ __forceinline__ cpair scal(cpair a, float s) { return {{kpmx::scal(a.v[0], s), kpmx::scal(a.v[1], s)}}; }
__device__ __forceinline__ fquad sub(fquad a, fquad b) {
    return {{a.v[0] - b.v[0], a.v[1] - b.v[1], a.v[2] - b.v[2], a.v[3] - b.v[3]}};
}
__device__ __forceinline__ cpair sub(cpair a, cpair b) {
    return {{kpmx::sub(a.v[0], b.v[0]), kpmx::sub(a.v[1], b.v[1])}};
}
using kpmx::fmac;
using kpmx::scal;
using kpmx::sub;
// sum of two elements (the uniform form adds the gathered elements before one multiplication)
__device__ __forceinline__ float plus(float a, float b) { return a + b; }
__device__ __forceinline__ double plus(double a, double b) { return a + b; }
template <class R> __device__ __forceinline__ cplx<R> plus(cplx<R> a, cplx<R> b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ dpair plus(dpair a, dpair b) { return {a.a + b.a, a.b + b.b}; }
__device__ __forceinline__ fquad plus(fquad a, fquad b) {
    return {{a.v[0] + b.v[0], a.v[1] + b.v[1], a.v[2] + b.v[2], a.v[3] + b.v[3]}};
}
__device__ __forceinline__ cpair plus(cpair a, cpair b) { return {{plus(a.v[0], b.v[0]), plus(a.v[1], b.v[1])}}; }

// matrix value times element
__device__ __forceinline__ float product(float a, float b) { return a * b; }
__device__ __forceinline__ double product(double a, double b) { return a * b; }
template <class R> __device__ __forceinline__ cplx<R> product(cplx<R> a, cplx<R> b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ dpair product(double a, dpair b) { return {a * b.a, a * b.b}; }
__device__ __forceinline__ fquad product(float a, fquad b) { return {{a * b.v[0], a * b.v[1], a * b.v[2], a * b.v[3]}}; }
__device__ __forceinline__ cpair product(cf32 a, cpair b) { return {{product(a, b.v[0]), product(a, b.v[1])}}; }

// the sums of one element, kind-major: |x|^2 of every column, then conj(y) x (real parts, then
// imaginary parts), added to s[kinds * cols]
__device__ __forceinline__ void add_sums(float y, float x, double* s) {
    s[0] += double(x) * double(x);
    s[1] += double(y) * double(x);
}
__device__ __forceinline__ void add_sums(double y, double x, double* s) {
    s[0] += x * x;
    s[1] += y * x;
}
__device__ __forceinline__ void add_sums(dpair y, dpair x, double* s) {
    s[0] += x.a * x.a;
    s[1] += x.b * x.b;
    s[2] += y.a * x.a;
    s[3] += y.b * x.b;
}
__device__ __forceinline__ void add_sums(fquad y, fquad x, double* s) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        s[c] += double(x.v[c]) * double(x.v[c]);
        s[4 + c] += double(y.v[c]) * double(x.v[c]);
    }
}
template <class R>
__device__ __forceinline__ void add_sums(cplx<R> y, cplx<R> x, double* s) {
    s[0] += sqabs(x);
    const d2 p = cdot(y, x);
    s[1] += p.re;
    s[2] += p.im;
}
__device__ __forceinline__ void add_sums(cpair y, cpair x, double* s) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        s[c] += sqabs(x.v[c]);
        const d2 p = cdot(y.v[c], x.v[c]);
        s[2 + c] += p.re;
        s[4 + c] += p.im;
    }
}

// ------------------------------------------------------------------------------ the steps
template <int N, class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
// f(0), ..., f(N - 1) with constant arguments: arrays indexed by them stay in registers
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

// LDS of one workgroup: two of them on a CU's 160 KB
constexpr size_t LDS_BYTES = 160 * 1024 / 2;
// Shape of the kernel for an element type, row width, matrix form and row length (FEW: at most four
// entries).
template <class E, int EW, int FORM, bool FEW>
struct shape {
    using V = typename elem<E>::value;
    static constexpr int NS = elem<E>::kinds * elem<E>::cols;  // sums of an element
    static constexpr int sums = 2 * (elem<E>::kinds - 1) * elem<E>::cols;  // most of any collection
    // of few entries, rows of one small element keep them in registers, wider rows in LDS; longer
    // rows read them from L1 and L2 in every step
    static constexpr bool narrow = EW * sizeof(E) < 16;
    // 16 waves where 64 registers do (fp64 block of 32 on 1.05 M sites, 258 moments: 8.4 ms against
    // 9.6 ms with 8 waves); 8 waves where a thread needs more: eight fp32 sums (6.5 against 8.7 ms on
    // 1.2 M sites), stored values (complex128, 16 vectors, 512 k sites: 6.4 against 6.7 ms), entries
    // in registers (one fp64 vector, 2.1 M sites, 514 moments: 1.4 ms; 16 waves hold 4096 rows only),
    // long rows (19 entries, 123 k rows, 24 vectors, 514 moments: 7.6 against 11 ms)
    static constexpr int threads = FEW && FORM != CHAIN_STD && !narrow && NS <= 4 ? 1024 : 512;
    static constexpr int waves = threads / 64;
    static constexpr int waves_per_simd = 2 * waves / 4;  // two workgroups per CU
    // LDS bytes of a local row's entries: local columns, codes, diagonal
    static constexpr size_t row_entries = narrow || !FEW ? 0 : 8 + (FORM == CHAIN_TABLE ? 4 : 0) + (FORM != CHAIN_STD ? sizeof(V) : 0);
    // LDS beside the rows: two buffers of per-wave sums, the zero row, the ring counts, the value table
    static constexpr size_t fixed = 2 * waves * sums * EW * sizeof(double) + (EW * sizeof(E) + 31) / 16 * 16 + 64 +
                                    (FORM == CHAIN_TABLE ? 256 * sizeof(V) : 0);
    static constexpr int max_items = !FEW ? 8 : narrow ? 10 : 20;  // registers
    static constexpr int fit(int items) {  // rows that `items` items per thread leave LDS for
        const size_t entries = (size_t)items * threads / EW * row_entries;
        const int rows = entries + fixed >= LDS_BYTES ? 0 : (int)((LDS_BYTES - fixed - entries) / (EW * sizeof(E)));
        return rows < items * threads / EW ? rows : items * threads / EW;
    }
    static constexpr int best_items() {
        int best = 1;
        for (int i = 1; i <= max_items && (size_t)i * threads * sizeof(E) <= LDS_BYTES; ++i)
            if (fit(i) > fit(best)) best = i;
        return best;
    }
    static constexpr int items = best_items();  // per thread
    static constexpr int rows = fit(items);     // local rows a workgroup holds
    static constexpr int entry_rows = items * threads / EW;
};

template <class E>
struct ChainArgs {
    using value = typename elem<E>::value;
    const int32_t* perm;  // matrix row of every plan row (null: the same)
    const int32_t* tile_begin;
    const int32_t* ring;
    const int32_t* ext;
    int64_t ext_stride;
    const ushort4* lidx;
    const uint32_t* codes;
    const value* vals;
    const value* diag;
    const value* table;
    const int32_t* tile_table;  // first table entry of every tile (null: 0)
    int table_size;
    int groups, rows_x, rows_y;
    int64_t ntiles;
    const E* x;
    int64_t ldx, ldprev, ldout;  // in elements
    const E* xprev;
    E* out1;
    E* out2;
    double* partials;
    int64_t x_group, w_group, partials_group;  // from one column group to the next
    int steps, first;
    // the other collections (see ChainLaunch)
    const E* w;
    E* panel;
    int64_t panel_col, panel_step;
    const ushort4* op_lidx;
    const value* op_vals;
    int op_groups, op_rows;
    const int32_t* mark;
    E* mark_out;
    int64_t mark_stride;
};

// p[i] with a uniform p: a scalar base and a 32-bit lane offset
template <class P>
__device__ __forceinline__ P& at(P* p, unsigned i) {
    using byte = std::conditional_t<std::is_const_v<P>, const char, char>;
    return *reinterpret_cast<P*>(reinterpret_cast<byte*>(p) + (size_t)(i * (unsigned)sizeof(P)));
}

// the sums of <w| on one element: conj(w) x (real, imaginary part), then conj(w) y
template <class T>
__device__ __forceinline__ void add_dots(T w, T y, T x, double* s) {
    constexpr int P = elem<T>::kinds == 3 ? 2 : 1;
    const d2 a = cdot(w, x), b = cdot(w, y);
    s[0] += a.re;
    s[P] += b.re;
    if constexpr (P == 2) {
        s[1] += a.im;
        s[3] += b.im;
    }
}

// element of one column stored by the column (E of several columns: column i of the element)
template <class E>
__device__ __forceinline__ auto column_of(const E& e, int) { return e; }
__device__ __forceinline__ double column_of(const dpair& e, int i) { return i ? e.b : e.a; }
__device__ __forceinline__ float column_of(const fquad& e, int i) { return e.v[i]; }
__device__ __forceinline__ cf32 column_of(const cpair& e, int i) { return e.v[i]; }

// v plus v of another lane of the same row of 16 (DPP)
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
    union { double d; int i[2]; } a, b;
    a.d = v;
    b.i[0] = __builtin_amdgcn_update_dpp(0, a.i[0], CTRL, 0xF, 0xF, true);
    b.i[1] = __builtin_amdgcn_update_dpp(0, a.i[1], CTRL, 0xF, 0xF, true);
    return v + b.d;
}

// Halves of the wave (H = 32) or of each half (H = 16): the lower lanes get a's sum over both, the
// upper lanes b's.  One exchange halves two values at once, without selects.
template <int H>
__device__ __forceinline__ double fold(double a, double b) {
    union { double d; unsigned i[2]; } p, q;
    p.d = a;
    q.d = b;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const auto r = H == 32 ? __builtin_amdgcn_permlane32_swap(p.i[w], q.i[w], false, false)
                               : __builtin_amdgcn_permlane16_swap(p.i[w], q.i[w], false, false);
        p.i[w] = r[0];
        q.i[w] = r[1];
    }
    return p.d + q.d;
}

// Sums of s over the lanes of the wave with the same lane % EW, to red[value * EW + lane % EW]: two
// folds leave the row of 16 lanes number r with value 4 i + {0, 2, 1, 3}[r] (a fold puts its second
// argument in the upper lanes), rotations inside the rows (DPP) finish.
template <int NS, int EW>
__device__ __forceinline__ void wave_sums(const double* s, double* red) {
    const int lane = threadIdx.x & 63;
    const int r = lane >> 4, v = (r >> 1) | ((r & 1) << 1);
    static_for<(NS + 3) / 4>([&](auto group) {
        constexpr int I = decltype(group)::value * 4;
        auto value = [&](int i) { return i < NS ? s[i < NS ? i : 0] : 0.0; };
        double t = fold<16>(fold<32>(value(I), value(I + 1)), fold<32>(value(I + 2), value(I + 3)));
        t = dpp_add<0x128>(t);                       // row_ror:8
        if constexpr (EW <= 4) t = dpp_add<0x124>(t);  // row_ror:4
        if constexpr (EW <= 2) t = dpp_add<0x122>(t);
        if constexpr (EW <= 1) t = dpp_add<0x121>(t);
        if ((lane & 15) < EW && I + v < NS) red[(I + v) * EW + lane % EW] = t;
    });
}

// W: entries per row (3 or 4 unrolled; 0: groups of four in a loop).  MODE: what a step leaves beside
// the vectors (CHAIN_SUMS ... CHAIN_MARKS, see ChainLaunch).
template <class E, int EW, int FORM, int W, int MODE>
__global__ __launch_bounds__((shape<E, EW, FORM, (W > 0)>::threads), (shape<E, EW, FORM, (W > 0)>::waves_per_simd))
void k_chain(ChainArgs<E> a) {
    using V = typename elem<E>::value;
    using real = typename elem<E>::real;
    using S = shape<E, EW, FORM, (W > 0)>;
    constexpr int IT = S::items, THREADS = S::threads, WAVES = S::waves;
    constexpr bool SUMS = MODE == CHAIN_SUMS || MODE == CHAIN_DOTS;
    // 32-bit sums run in the order of the stored row, diagonal in its place, as the single steps do: the
    // vectors are theirs bit for bit (in 64 bits the order is free)
    constexpr bool ORDERED = sizeof(real) == 4;
    constexpr int NS = MODE == CHAIN_DOTS ? 2 * (elem<E>::kinds - 1) : SUMS ? S::NS : 1;
    // items loaded together, as many as the registers allow (fp32 block of 32 on 1.2 M sites, 258
    // moments: 6.4 ms with four, 6.85 ms with two)
    constexpr int LD = THREADS == 512 && EW * sizeof(E) >= 16 ? 4 : 2;
    constexpr bool KEEP = W > 0 && S::narrow;  // entries in registers
    constexpr bool LDS_ENTRIES = W > 0 && !S::narrow;
    extern __shared__ __align__(16) char smem[];
    E* X = reinterpret_cast<E*>(smem);  // the rows, then the zero row
    char* lds = smem + (size_t)S::rows * EW * sizeof(E) + (EW * sizeof(E) + 15) / 16 * 16;
    lds = smem + ((lds - smem) + 15) / 16 * 16;
    double* red = reinterpret_cast<double*>(lds);
    lds += 2 * WAVES * S::sums * EW * sizeof(double);
    int* rings = reinterpret_cast<int*>(lds);
    lds += 64;
    V* tab = reinterpret_cast<V*>(lds);
    if constexpr (FORM == CHAIN_TABLE) lds += 256 * sizeof(V);
    ushort4* sid = reinterpret_cast<ushort4*>(lds + (FORM == CHAIN_STD ? 0 : S::entry_rows * sizeof(V)));
    V* sdiag = reinterpret_cast<V*>(lds);
    uint32_t* scode = reinterpret_cast<uint32_t*>(sid + S::entry_rows);

    // tiles of one eighth of the rows on one XCD: neighbours' halo rows stay in its L2
    const int64_t per = (a.ntiles + 7) / 8;
    int64_t turn = blockIdx.x / 8;
    if constexpr (MODE == CHAIN_SUMS)
        for (; turn >= per; turn -= per) {  // column groups side by side
            a.x += a.x_group;
            a.xprev += a.w_group;
            a.out1 += a.w_group;
            a.out2 += a.w_group;
            a.partials += a.partials_group;
        }
    const int64_t t = (int64_t)(blockIdx.x % 8) * per + turn;
    if (t >= a.ntiles) return;
    const int tid = threadIdx.x, c = tid % EW;
    const unsigned trow = (unsigned)tid / EW;
    const E* Xc = X + c;  // entries hold a row's first item
    const int64_t r0 = a.tile_begin[t];
    const int own = (int)(a.tile_begin[t + 1] - r0);
    const int32_t* rg = a.ring + t * (CHAIN_MAX_STEPS + 1);
    const int32_t* halo = a.ext + t * a.ext_stride;
    const int nx = rg[a.steps] * EW, ny = rg[a.steps - 1] * EW, nown = own * EW;

    // own rows first, then the halo; r_{k-1} straight to registers
    E y[IT];
    static_for<(IT + LD - 1) / LD>([&](auto chunk) {
        constexpr int I0 = decltype(chunk)::value * LD, N = I0 + LD < IT ? LD : IT - I0;
        E xv[N];
        int32_t g[N];
        static_for<N>([&](auto u) {
            const int first = (I0 + u) * THREADS;  // item of thread 0
            g[u] = (int32_t)r0 + (int32_t)trow + first / EW;
            if (tid >= nown - first && tid < nx - first) g[u] = at(halo + (first / EW - own), trow);
            // the first launch reads the caller's vectors, in the matrix's row order
            if (a.first && a.perm && tid < nx - first) g[u] = a.perm[g[u]];
        });
        static_for<N>([&](auto u) {
            xv[u] = make_zero<E>();
            if (tid < nx - (I0 + u) * THREADS) xv[u] = a.x[(int64_t)g[u] * a.ldx + c];
        });
        static_for<N>([&](auto u) {
            y[I0 + u] = make_zero<E>();
            if (!a.first && tid < ny - (I0 + u) * THREADS) y[I0 + u] = a.xprev[(int64_t)g[u] * a.ldprev + c];
        });
        static_for<N>([&](auto u) {
            if (tid < nx - (I0 + u) * THREADS) X[tid + (I0 + u) * THREADS] = xv[u];
        });
    });
    const int first_value = FORM != CHAIN_STD && a.tile_table ? a.tile_table[t] : 0;
    if constexpr (FORM == CHAIN_TABLE)
        if (tid < 256 && first_value + tid < a.table_size) tab[tid] = a.table[first_value + tid];
    if (tid < EW) X[a.rows_x * EW + tid] = make_zero<E>();
    if (tid <= a.steps) rings[tid] = rg[tid];
    const ushort4* lidx = a.lidx + t * a.groups * a.rows_y;
    const uint32_t* codes = a.codes + t * a.groups * a.rows_y;
    const V* vals = a.vals + t * 4 * a.groups * a.rows_y;
    const V* diag = a.diag + t * a.rows_y;
    ushort4 id[KEEP ? IT : 1];
    uint32_t code[KEEP && FORM == CHAIN_TABLE ? IT : 1];
    V dg[KEEP && FORM != CHAIN_STD ? IT : 1];
    if constexpr (KEEP)
        static_for<IT>([&](auto it) {
            const unsigned r = it * (THREADS / EW);
            if (it * THREADS >= ny) return;
            id[it] = at(lidx + r, trow);
            if constexpr (FORM == CHAIN_TABLE) code[it] = at(codes + r, trow);
            if constexpr (FORM != CHAIN_STD) dg[it] = at(diag + r, trow);
        });
    if constexpr (LDS_ENTRIES)
        for (int r = tid; r < a.rows_y; r += THREADS) {
            sid[r] = lidx[r];
            if constexpr (FORM == CHAIN_TABLE) scode[r] = codes[r];
            if constexpr (FORM != CHAIN_STD) sdiag[r] = diag[r];
        }
    V uniform = zero(V{});
    if constexpr (FORM == CHAIN_UNIFORM)
        if (first_value + 1 < a.table_size) uniform = a.table[first_value + 1];
    __syncthreads();

    // the tile's sums of step j, added up in wave order by one wave while the others go on
    auto store_sums = [&](int j) {
        const int i = tid & 63;
        if (tid / 64 != j % WAVES || i >= NS * EW) return;
        const double* rw = red + (j & 1) * WAVES * NS * EW + i;
        double v = rw[0];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v += rw[w * NS * EW];
        a.partials[((int64_t)(j - 1) * a.ntiles + t) * (NS * EW) + i] = v;
    };
    auto matrix_row = [&](unsigned row) -> int64_t {
        const int64_t g = r0 + row + trow;
        return a.perm ? a.perm[g] : g;
    };
    // row `row` (of thread 0) of the panel's step p, every column of the element to its own panel
    auto to_panel = [&](const E& e, int p, int row) {
        using T = decltype(column_of(e, 0));
        T* o = reinterpret_cast<T*>(a.panel) + p * a.panel_step + r0 + row + trow;
        static_for<elem<E>::cols>([&](auto i) { o[(int64_t)(c * elem<E>::cols + i) * a.panel_col] = column_of(e, i); });
    };
    const ushort4* op_lidx = a.op_lidx + t * a.op_groups * a.op_rows;
    const V* op_vals = a.op_vals + t * 4 * a.op_groups * a.op_rows;
    for (int j = 1; j <= a.steps; ++j) {
        unsigned again = 0;
        asm volatile("" : "+s"(again));
        const int act = __builtin_amdgcn_readfirstlane(rings[a.steps - j]) * EW;
        const real hs = (a.first && j == 1) ? real(0.5) : real(1);
        if constexpr (SUMS)
            if (j > 1) store_sums(j - 1);
        double s[NS] = {};
        static_for<IT>([&](auto item) {
            constexpr int it = decltype(item)::value;
            if (it * THREADS >= act) return;
            // lanes past the end compute on padding (LDS and entry arrays reach that far); their
            // results are never read.  What is not in registers or LDS is read again in every step
            // (L1, L2): hoisted out of the loop it would spill.
            constexpr int row = it * (THREADS / EW);  // of thread 0
            const unsigned r = row + again;
            E h = make_zero<E>();
            V d = zero(V{});
            const uint16_t self = (uint16_t)((row + trow) * EW);
            auto entry = [&](uint16_t l, V v, bool first) {
                const E xg = Xc[l];
                if constexpr (FORM == CHAIN_UNIFORM && !ORDERED) {
                    h = first ? xg : plus(h, xg);
                } else {
                    if constexpr (ORDERED && FORM != CHAIN_STD) v = l == self ? d : v;
                    h = first && !ORDERED ? product(v, xg) : fmac(v, xg, h);
                }
            };
            if constexpr (W > 0) {
                ushort4 l;
                uint32_t cd = 0;
                if constexpr (KEEP) {
                    l = id[it];
                    if constexpr (FORM == CHAIN_TABLE) cd = code[it];
                    if constexpr (FORM != CHAIN_STD) d = dg[it];
                } else {
                    l = sid[row + trow];
                    if constexpr (FORM == CHAIN_TABLE) cd = scode[row + trow];
                    if constexpr (FORM != CHAIN_STD) d = sdiag[row + trow];
                }
                V v[4] = {};
                static_for<W>([&](auto k) {
                    if constexpr (FORM == CHAIN_STD) v[k] = at(vals + ((unsigned)(k * a.rows_y) + r), trow);
                    if constexpr (FORM == CHAIN_TABLE) v[k] = tab[(cd >> (8 * k)) & 255];
                    if constexpr (FORM == CHAIN_UNIFORM) v[k] = uniform;
                });
                entry(l.x, v[0], true);
                entry(l.y, v[1], false);
                entry(l.z, v[2], false);
                if constexpr (W > 3) entry(l.w, v[3], false);
            } else {
                ushort4 next = at(lidx + r, trow);
                uint32_t next_code = FORM == CHAIN_TABLE ? at(codes + r, trow) : 0u;
                if constexpr (FORM != CHAIN_STD) d = at(diag + r, trow);
                for (int g = 0; g < a.groups; ++g) {
                    const ushort4 l = next;
                    const uint32_t cd = next_code;
                    const unsigned o = (unsigned)(g * a.rows_y) + r;
                    if (g + 1 < a.groups) {
                        next = at(lidx + (o + a.rows_y), trow);
                        if constexpr (FORM == CHAIN_TABLE) next_code = at(codes + (o + a.rows_y), trow);
                    }
                    V v[4] = {};
                    static_for<4>([&](auto k) {
                        if constexpr (FORM == CHAIN_STD) v[k] = at(vals + ((unsigned)((4 * g + k) * a.rows_y) + r), trow);
                        if constexpr (FORM == CHAIN_TABLE) v[k] = tab[(cd >> (8 * k)) & 255];
                        if constexpr (FORM == CHAIN_UNIFORM) v[k] = uniform;
                    });
                    entry(l.x, v[0], false);
                    entry(l.y, v[1], false);
                    entry(l.z, v[2], false);
                    entry(l.w, v[3], false);
                }
            }
            const E xi = X[tid + it * THREADS];
            if constexpr (FORM == CHAIN_UNIFORM && !ORDERED) h = product(uniform, h);
            if constexpr (FORM != CHAIN_STD && !ORDERED) h = fmac(d, xi, h);
            y[it] = sub(scal(h, hs), y[it]);
            if constexpr (MODE == CHAIN_SUMS)
                if (tid < nown - it * THREADS) add_sums(y[it], xi, s);
            if constexpr (MODE == CHAIN_DOTS)
                if (tid < nown - it * THREADS) add_dots(a.w[matrix_row(row + again)], y[it], xi, s);
            if constexpr (MODE == CHAIN_PANEL)
                if (tid < nown - it * THREADS) to_panel(y[it], j, row);
            if constexpr (MODE == CHAIN_PANEL_OP)
                if (tid < nown - it * THREADS) {
                    E o = make_zero<E>();
                    for (int g = 0; g < a.op_groups; ++g) {
                        const unsigned q = (unsigned)(g * a.op_rows) + r;
                        const ushort4 l = at(op_lidx + q, trow);
                        const uint16_t id[4] = {l.x, l.y, l.z, l.w};
                        static_for<4>([&](auto k) {
                            o = fmac(at(op_vals + ((unsigned)((4 * g + k) * a.op_rows) + r), trow), Xc[id[k]], o);
                        });
                    }
                    to_panel(scal(o, hs), j - 1, row);
                }
            if constexpr (MODE == CHAIN_MARKS)
                if (tid < nown - it * THREADS) {
                    const int m = a.mark[matrix_row(row + again)];
                    if (m >= 0) a.mark_out[m * a.mark_stride + j] = y[it];
                }
        });
        if constexpr (SUMS) wave_sums<NS, EW>(s, red + ((j & 1) * WAVES + tid / 64) * NS * EW);
        __syncthreads();
        if (j == a.steps) break;
        static_for<IT>([&](auto it) {
            if (tid < act - it * THREADS) {
                const E xi = X[tid + it * THREADS];
                X[tid + it * THREADS] = y[it];
                y[it] = xi;
            }
        });
        __syncthreads();
    }
    if constexpr (SUMS) store_sums(a.steps);
    static_for<IT>([&](auto it) {
        if (tid < nown - it * THREADS) {
            const int64_t o = (r0 + it * (THREADS / EW) + trow) * a.ldout + c;
            a.out2[o] = y[it];
            if (a.steps > 1) a.out1[o] = X[tid + it * THREADS];
        }
    });
}

// Elements of the rows of a scalar type: f(E{}, integral EW) for `cols` vectors (-1: no such layout)
template <class T, class F>
int with_layout(int cols, F&& f) {
    using one = std::integral_constant<int, 1>;
    using two = std::integral_constant<int, 2>;
    using four = std::integral_constant<int, 4>;
    if constexpr (std::is_same_v<T, float>) {
        if (cols == 1) return f(float{}, one{});
        if (cols == 2) return f(float{}, two{});
        if (cols == 4) return f(fquad{}, one{});
        if (cols == 8) return f(fquad{}, two{});
        if (cols == 16) return f(fquad{}, four{});
    } else if constexpr (std::is_same_v<T, cf64>) {
        if (cols == 1) return f(cf64{}, one{});
        if (cols == 2) return f(cf64{}, two{});
        if (cols == 4) return f(cf64{}, four{});
    } else {
        using pair = std::conditional_t<std::is_same_v<T, double>, dpair, cpair>;
        if (cols == 1) return f(T{}, one{});
        if (cols == 2) return f(pair{}, one{});
        if (cols == 4) return f(pair{}, two{});
        if (cols == 8) return f(pair{}, four{});
    }
    return -1;
}
template <class F>
int with_layout(int scalar, int cols, F&& f) {
    switch (scalar) {
        case 0: return with_layout<float>(cols, f);
        case 1: return with_layout<double>(cols, f);
        case 2: return with_layout<cf32>(cols, f);
        default: return with_layout<cf64>(cols, f);
    }
}

// Lets a kernel use more than the default 64 KB of LDS, once per device.
inline bool allow_lds(const void* kernel, size_t bytes, std::atomic<uint64_t>& allowed) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return false;
    const uint64_t bit = uint64_t(1) << (device & 63);
    if (allowed.load(std::memory_order_acquire) & bit) return true;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) return false;
    allowed.fetch_or(bit, std::memory_order_release);
    return true;
}

template <class E, int EW, int FORM, int W, int MODE>
int launch_form(const ChainLaunch& L, hipStream_t s) {
    using V = typename elem<E>::value;
    const ChainPlan& P = *L.plan;
    ChainArgs<E> a{};
    a.perm = L.m.perm;
    a.tile_begin = P.tile_begin;
    a.ring = P.ring;
    a.ext = P.ext;
    a.ext_stride = P.ext_stride;
    a.lidx = P.lidx;
    a.codes = P.codes;
    a.vals = static_cast<const V*>(P.vals);
    a.diag = static_cast<const V*>(P.diag);
    a.table = static_cast<const V*>(L.m.table);
    a.tile_table = P.tile_table;
    a.table_size = L.m.table_size;
    a.groups = P.groups;
    a.rows_x = P.rows_x;
    a.rows_y = P.rows_y;
    a.ntiles = P.ntiles;
    a.x = static_cast<const E*>(L.x);
    a.ldx = L.ldx / elem<E>::cols;
    a.ldprev = L.ldprev ? L.ldprev / elem<E>::cols : EW;
    a.ldout = L.ldout ? L.ldout / elem<E>::cols : EW;
    a.xprev = static_cast<const E*>(L.xprev);
    a.out1 = static_cast<E*>(L.out1);
    a.out2 = static_cast<E*>(L.out2);
    a.partials = L.partials;
    a.x_group = L.x_group / elem<E>::cols;
    a.w_group = L.w_group / elem<E>::cols;
    a.partials_group = L.partials_group;
    a.steps = L.steps;
    a.first = L.first;
    a.w = static_cast<const E*>(L.w);
    a.panel = static_cast<E*>(L.panel);
    a.panel_col = L.panel_col;
    a.panel_step = L.panel_step;
    if (L.op) {
        a.op_lidx = L.op->lidx;
        a.op_vals = static_cast<const V*>(L.op->vals);
        a.op_groups = L.op->groups;
        a.op_rows = L.op->rows;
    }
    a.mark = L.mark;
    a.mark_out = static_cast<E*>(L.mark_out);
    a.mark_stride = L.mark_stride;
    auto kernel = k_chain<E, EW, FORM, W, MODE>;
    static std::atomic<uint64_t> allowed{0};  // devices
    if (!allow_lds(reinterpret_cast<const void*>(kernel), LDS_BYTES, allowed)) return -1;
    const int64_t grid = (P.ntiles + 7) / 8 * 8 * L.col_groups;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(shape<E, EW, FORM, (W > 0)>::threads), LDS_BYTES, s, a);
    return 0;
}

template <class E, int EW, int MODE>
int launch_mode(const ChainLaunch& L, hipStream_t s) {
    const int w = L.plan->groups > 1 ? 0 : L.plan->width <= 3 ? 3 : 4;
    auto by_width = [&](auto form) {
        constexpr int F = decltype(form)::value;
        if (w == 3) return launch_form<E, EW, F, 3, MODE>(L, s);
        if (w == 4) return launch_form<E, EW, F, 4, MODE>(L, s);
        return launch_form<E, EW, F, 0, MODE>(L, s);
    };
    switch (L.m.form()) {
        case CHAIN_STD: return by_width(std::integral_constant<int, CHAIN_STD>{});
        case CHAIN_TABLE: return by_width(std::integral_constant<int, CHAIN_TABLE>{});
        default: return by_width(std::integral_constant<int, CHAIN_UNIFORM>{});
    }
}

// the collections beside the diagonal sums exist for one column and, panels, for the widest rows
template <class E, int EW>
int launch_elem(const ChainLaunch& L, hipStream_t s) {
    constexpr bool one = EW * elem<E>::cols == 1, widest = EW == 4;
    if (L.mode == CHAIN_SUMS) return launch_mode<E, EW, CHAIN_SUMS>(L, s);
    if constexpr (one) {
        if (L.mode == CHAIN_DOTS) return launch_mode<E, EW, CHAIN_DOTS>(L, s);
        if (L.mode == CHAIN_MARKS) return launch_mode<E, EW, CHAIN_MARKS>(L, s);
    }
    if constexpr (one || widest) {
        if (L.mode == CHAIN_PANEL) return launch_mode<E, EW, CHAIN_PANEL>(L, s);
        if (L.mode == CHAIN_PANEL_OP) return launch_mode<E, EW, CHAIN_PANEL_OP>(L, s);
    }
    return -1;
}

}  // namespace
}  // namespace kpmx
