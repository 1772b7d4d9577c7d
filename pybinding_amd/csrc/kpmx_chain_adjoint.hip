// The chained backward recurrence of the adjoint gradient: several reverse steps per launch, on the
// plans of kpmx_chain.hip.
//
// A reverse step (k_adjoint_sellb) gathers lambda_j+1 and v_j, reads lambda_j+2 and v_j+1, writes
// lambda_j and v_j-1 and reads and writes one gradient value per stored entry: about 830 bytes per
// row of 16 fp64 columns, and it runs at the card's memory rate.  Here v and lambda of a tile and its
// halo stay in LDS for K steps, v_j+1, lambda_j+2 and the gradients of the tile's own rows (which no
// other workgroup touches) in registers: two times four passes and one gradient update per K steps.
// 305 k strained sites, 16 fp64 columns, 258 moments, checkpoints every 64: 129 steps of 47 us before,
// 34 launches per group of four columns of 31 us now (K = 4; 20 us of them memory, 20 MB of gradients
// and 80 MB of vectors out of the Infinity Cache, the rest LDS gathers and fp64 arithmetic).  Taken from
// measurements there: groups of four columns (two workgroups of 1100 rows per CU) rather than eight
// (600 rows, K = 4: 87 us; one workgroup of 1200 rows per CU: 75 us, nothing overlaps its loads);
// packed work vectors, one group after the other (all groups side by side on the 16-column blocks:
// 169 us for 4 x 39); values re-read from L2 in every step (in LDS they would take a quarter of the
// tile; loaded one item ahead, the 128 registers spill: 33.7 us); row-major gradients, which the lanes
// of a row load and store side by side.
#include "kpmx_chain_step.hpp"

#include <algorithm>

namespace kpmx {
namespace {

template <class E, int EW>
struct adjoint_shape {
    static constexpr int threads = 512;
    static constexpr size_t lds = LDS_BYTES;
    static constexpr int items = 5;      // of each vector per thread (registers)
    static constexpr int own_items = 3;  // of the tile's own rows: their gradients are registers, too
    static constexpr int entry_rows = items * threads / EW;
    static constexpr size_t fixed = 2 * EW * sizeof(E) + 64 + 64;  // zero rows, ring counts, alignment
    static_assert((CHAIN_MAX_STEPS + 1) * sizeof(int) <= 64, "ring counts");
    static constexpr int fit = (int)((lds - fixed - entry_rows * sizeof(ushort4)) / (2 * EW * sizeof(E)));
    static constexpr int rows = fit < entry_rows ? fit : entry_rows;
    static constexpr int own_rows = own_items * threads / EW;
};

template <class E>
struct AdjointChainArgs {
    using value = typename elem<E>::value;
    const int32_t* tile_begin;
    const int32_t* ring;
    const int32_t* ext;
    int64_t ext_stride;
    const ushort4* lidx;
    const value* vals;
    int rows_x, rows_y;
    int64_t ntiles;
    int64_t ldv, ldlam;  // of v and v_next, of lam_out, in elements (the others: EW)
    const E* v;
    const E* v_next;
    const E* lam;
    const E* lam_next;
    E* v_out;
    E* v_next_out;
    E* lam_out;
    E* lam_next_out;
    double* grad;  // [row][4]
    int steps;
    double ca[CHAIN_MAX_STEPS], chv[CHAIN_MAX_STEPS], cg[CHAIN_MAX_STEPS];
};

// one element's share of sum over columns of a[c] b[c], products in the columns' precision
__device__ __forceinline__ double col_products(dpair a, dpair b) { return a.a * b.a + a.b * b.b; }
__device__ __forceinline__ double col_products(fquad a, fquad b) {
    return ((double)(a.v[0] * b.v[0]) + (double)(a.v[1] * b.v[1])) + ((double)(a.v[2] * b.v[2]) + (double)(a.v[3] * b.v[3]));
}

// computes a result where it stands: the compiler would put the arithmetic of all items off to the end
// of the step, with everything they gathered in registers (400 to 700 bytes of spills per lane)
__device__ __forceinline__ void pin(double& a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ void pin(dpair& e) { asm volatile("" : "+v"(e.a), "+v"(e.b)); }
__device__ __forceinline__ void pin(fquad& e) { asm volatile("" : "+v"(e.v[0]), "+v"(e.v[1]), "+v"(e.v[2]), "+v"(e.v[3])); }

template <class E, int EW, int W>
__global__ __launch_bounds__((adjoint_shape<E, EW>::threads), 4) void k_chain_adjoint(AdjointChainArgs<E> a) {
    using V = typename elem<E>::value;
    using S = adjoint_shape<E, EW>;
    constexpr int IT = S::items, OI = S::own_items, THREADS = S::threads;
    extern __shared__ __align__(16) char smem[];
    E* Xv = reinterpret_cast<E*>(smem);  // the rows, then the zero row; the same for lambda
    E* Xl = Xv + (S::rows + 1) * EW;
    ushort4* sid = reinterpret_cast<ushort4*>(Xl + (S::rows + 1) * EW);
    int* rings = reinterpret_cast<int*>(sid + S::entry_rows);

    const int64_t per = (a.ntiles + 7) / 8;  // tiles of one eighth of the rows on one XCD
    const int64_t t = (int64_t)(blockIdx.x % 8) * per + blockIdx.x / 8;
    if (t >= a.ntiles) return;
    const int tid = threadIdx.x, c = tid % EW;
    const unsigned trow = (unsigned)tid / EW;
    const int64_t r0 = a.tile_begin[t];
    const int own = (int)(a.tile_begin[t + 1] - r0);
    const int32_t* rg = a.ring + t * (CHAIN_MAX_STEPS + 1);
    const int32_t* halo = a.ext + t * a.ext_stride;
    const int nx = rg[a.steps] * EW, ny = rg[a.steps - 1] * EW, nown = own * EW;

    const ushort4* lidx = a.lidx + t * a.rows_y;
    const V* vals = a.vals + t * 4 * a.rows_y;
    for (int r = tid; r < a.rows_y; r += THREADS) sid[r] = lidx[r];
    int32_t row_of[IT];
    static_for<IT>([&](auto it) {
        constexpr int first = decltype(it)::value * THREADS;
        row_of[it] = (int32_t)r0 + (int32_t)trow + first / EW;
        if (tid >= nown - first && tid < nx - first) row_of[it] = at(halo + (first / EW - own), trow);
    });
    E vn[IT], ln[IT], xv[IT], xl[IT];  // all loads in flight at once
    static_for<IT>([&](auto it) {
        xv[it] = xl[it] = make_zero<E>();
        if (tid < nx - it * THREADS) {
            xv[it] = a.v[(int64_t)row_of[it] * a.ldv + c];
            if (a.lam) xl[it] = a.lam[(int64_t)row_of[it] * EW + c];
        }
    });
    static_for<IT>([&](auto it) {
        vn[it] = ln[it] = make_zero<E>();
        if (tid < ny - it * THREADS) {
            vn[it] = a.v_next[(int64_t)row_of[it] * a.ldv + c];
            if (a.lam) ln[it] = a.lam_next[(int64_t)row_of[it] * EW + c];
        }
    });
    static_for<IT>([&](auto it) {
        if (tid < nx - it * THREADS) {
            Xv[tid + it * THREADS] = xv[it];
            Xl[tid + it * THREADS] = xl[it];
        }
    });
    if (tid < EW) {
        Xv[a.rows_x * EW + tid] = make_zero<E>();
        Xl[a.rows_x * EW + tid] = make_zero<E>();
    }
    if (tid <= a.steps) rings[tid] = rg[tid];
    // lane c holds the sums of entries c, c + EW, ... so far
    double g[OI][W];
    static_for<OI>([&](auto it) {
        double old[(W + EW - 1) / EW];
        static_for<(W + EW - 1) / EW>([&](auto m) {
            double o = 0;
            if (tid < nown - it * THREADS) o = a.grad[(r0 + it * (THREADS / EW) + trow) * 4 + m * EW + c];
            old[m] = o;
        });
        static_for<W>([&](auto k) { g[it][k] = k % EW == c ? old[k / EW] : 0.0; });
    });
    __syncthreads();

    for (int j = 1; j <= a.steps; ++j) {
        unsigned again = 0;
        asm volatile("" : "+s"(again));  // the values are read again in every step: kept, they would spill
        const int act = __builtin_amdgcn_readfirstlane(rings[a.steps - j]) * EW;
        const V ca = (V)a.ca[j - 1], chv = (V)a.chv[j - 1], cg = (V)a.cg[j - 1];
        static_for<IT>([&](auto item) {
            constexpr int it = decltype(item)::value;
            constexpr int row = it * (THREADS / EW);
            if (it * THREADS >= act) return;
            // lanes past the end compute on padding, as in k_chain
            const ushort4 l4 = sid[row + trow];
            const uint16_t l[4] = {l4.x, l4.y, l4.z, l4.w};
            const E vo = Xv[tid + it * THREADS], lo = Xl[tid + it * THREADS];
            E acc_v = make_zero<E>(), acc_l = make_zero<E>();
            const E rf = fmac(cg, vo, lo);
            static_for<W>([&](auto k) {
                const V m = at(vals + ((unsigned)(k * a.rows_y) + row + again), trow);
                const E xv = Xv[l[k] + c], xl = Xl[l[k] + c];
                acc_l = fmac(m, xl, acc_l);
                acc_v = fmac(m, xv, acc_v);
                if constexpr (it < OI) {
                    g[it][k] += col_products(rf, xv);  // of lanes past the own rows: dropped below
                    pin(g[it][k]);
                }
            });
            E lnew = sub(acc_l, ln[it]);
            lnew = fmac(ca, vo, lnew);
            lnew = fmac(chv, acc_v, lnew);
            ln[it] = lnew;
            vn[it] = sub(acc_v, vn[it]);
            pin(ln[it]);
            pin(vn[it]);
        });
        if (j == a.steps) break;
        __syncthreads();
        static_for<IT>([&](auto it) {
            if (tid < act - it * THREADS) {
                const E v = Xv[tid + it * THREADS], l = Xl[tid + it * THREADS];
                Xv[tid + it * THREADS] = vn[it];
                Xl[tid + it * THREADS] = ln[it];
                vn[it] = v;
                ln[it] = l;
            }
        });
        __syncthreads();
    }
    static_for<IT>([&](auto it) {
        if (tid < nown - it * THREADS) {
            const int64_t row = r0 + it * (THREADS / EW) + trow, o = row * EW + c;
            if (a.v_out) {
                a.v_out[o] = vn[it];
                a.v_next_out[o] = Xv[tid + it * THREADS];
            }
            a.lam_out[row * a.ldlam + c] = ln[it];
            if (a.lam_next_out) a.lam_next_out[o] = Xl[tid + it * THREADS];
        }
    });
    // entry k of a row, summed over its EW lanes (quad permutes)
    static_for<OI>([&](auto it) {
        if (it * THREADS >= nown) return;  // uniform
        static_for<W>([&](auto k) {
            double s = g[it][k];
            if constexpr (EW >= 2) s = dpp_add<0xB1>(s);  // lane ^ 1
            if constexpr (EW >= 4) s = dpp_add<0x4E>(s);  // lane ^ 2
            if (k % EW == c && tid < nown - it * THREADS) a.grad[(r0 + it * (THREADS / EW) + trow) * 4 + k] = s;
        });
    });
}

template <class E, int EW, int W>
int launch_one(const AdjointChainLaunch& L, hipStream_t s) {
    using V = typename elem<E>::value;
    const ChainPlan& P = *L.plan;
    AdjointChainArgs<E> a{};
    a.tile_begin = P.tile_begin;
    a.ring = P.ring;
    a.ext = P.ext;
    a.ext_stride = P.ext_stride;
    a.lidx = P.lidx;
    a.vals = static_cast<const V*>(P.vals);
    a.rows_x = P.rows_x;
    a.rows_y = P.rows_y;
    a.ntiles = P.ntiles;
    a.ldv = L.ldv / elem<E>::cols;
    a.ldlam = L.ldlam / elem<E>::cols;
    a.v = static_cast<const E*>(L.v);
    a.v_next = static_cast<const E*>(L.v_next);
    a.lam = static_cast<const E*>(L.lam);
    a.lam_next = static_cast<const E*>(L.lam_next);
    a.v_out = static_cast<E*>(L.v_out);
    a.v_next_out = static_cast<E*>(L.v_next_out);
    a.lam_out = static_cast<E*>(L.lam_out);
    a.lam_next_out = static_cast<E*>(L.lam_next_out);
    a.grad = L.grad;
    a.steps = L.steps;
    for (int j = 0; j < L.steps; ++j) {
        a.ca[j] = L.ca[j];
        a.chv[j] = L.chv[j];
        a.cg[j] = L.cg[j];
    }
    auto kernel = k_chain_adjoint<E, EW, W>;
    constexpr int threads = adjoint_shape<E, EW>::threads;
    constexpr size_t lds = adjoint_shape<E, EW>::lds;
    static std::atomic<uint64_t> allowed{0};
    if (!allow_lds(reinterpret_cast<const void*>(kernel), lds, allowed)) return -1;
    kernel<<<dim3((unsigned)((P.ntiles + 7) / 8 * 8)), dim3(threads), lds, s>>>(a);
    return 0;
}

template <class F>
int with_adjoint_layout(int scalar, int cols, F&& f) {
    if (scalar == 0 && cols == 4) return f(fquad{}, std::integral_constant<int, 1>{});
    if (scalar == 0 && cols == 8) return f(fquad{}, std::integral_constant<int, 2>{});
    if (scalar == 1 && cols == 4) return f(dpair{}, std::integral_constant<int, 2>{});
    return -1;
}

// SELL-ordered sums of rows of at most four entries from row-major ones
__global__ __launch_bounds__(256) void k_adjoint_chain_grad(const double* rows, const int64_t* slice_ptr, const int32_t* slice_width,
                                                            int64_t n, double* grad) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, r = i >> 2;
    const int k = (int)i & 3;
    if (r < n && k < slice_width[r >> 6]) grad[slice_ptr[r >> 6] + k * 64 + (r & 63)] = rows[i];
}

}  // namespace

void launch_adjoint_chain_grad(const ChainMatrix& m, const double* rows, double* grad, hipStream_t s) {
    hipLaunchKernelGGL(k_adjoint_chain_grad, dim3((unsigned)((m.n * 4 + 255) / 256)), dim3(256), 0, s, rows, m.slice_ptr,
                       m.slice_width, m.n, grad);
}

int chain_adjoint_cols(int scalar, int vw) { return scalar == 0 ? std::min(vw, 8) : 4; }

int chain_adjoint_capacity(int scalar, int cols) {
    return with_adjoint_layout(scalar, cols, [](auto e, auto ew) { return adjoint_shape<decltype(e), decltype(ew)::value>::rows; });
}
int chain_adjoint_own_rows(int scalar, int cols) {
    return with_adjoint_layout(scalar, cols,
                               [](auto e, auto ew) { return adjoint_shape<decltype(e), decltype(ew)::value>::own_rows; });
}
int chain_adjoint_row_pad(int scalar, int cols) {
    return with_adjoint_layout(scalar, cols, [](auto e, auto ew) {
        return adjoint_shape<decltype(e), decltype(ew)::value>::threads / decltype(ew)::value;
    });
}

int launch_adjoint_chain(const AdjointChainLaunch& L, hipStream_t s) {
    if (!L.plan || L.steps < 1 || L.ldv < L.cols || L.ldlam < L.cols || L.steps > L.plan->steps || L.plan->groups != 1 || L.m.codes ||
        L.plan->tile_rows > chain_adjoint_own_rows(L.m.scalar, L.cols) ||
        L.plan->rows_x > chain_adjoint_capacity(L.m.scalar, L.cols))
        return -1;
    return with_adjoint_layout(L.m.scalar, L.cols, [&](auto e, auto ew) {
        using E = decltype(e);
        constexpr int EW = decltype(ew)::value;
        return L.plan->width <= 3 ? launch_one<E, EW, 3>(L, s) : launch_one<E, EW, 4>(L, s);
    });
}

}  // namespace kpmx
