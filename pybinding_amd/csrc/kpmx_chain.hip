// Plans and sums of the chained diagonal recurrence (kpmx_chain_step.hpp has the step kernel).
//
// A plan is built on the device, once per matrix and column width, since it has to pay for itself
// within one run: sampled halos of eight heights (30 to 70 us), breadth-first rings of every tile (45 to
// 150 us) and its entries in local columns (10 to 30 us), one workgroup per tile with its set of rows in
// LDS.  They are bound by the rings' dependent gathers.
#include "kpmx_chain_step.hpp"

#include <algorithm>

namespace kpmx {
namespace {

// ------------------------------------------------------------------------------ plan kernels
constexpr int PLAN_THREADS = 512;

// A set of at most `limit` rows in LDS: 2^bits >= 2 limit slots of linear probing.
struct RowSet {
    int32_t* keys;
    int bits;
    __device__ unsigned slot(int32_t row) const { return ((unsigned)row * 2654435761u) >> (32 - bits); }
    __device__ unsigned next(unsigned h) const { return (h + 1) & ((1u << bits) - 1); }
    __device__ void clear() {
        for (int i = threadIdx.x; i < 1 << bits; i += PLAN_THREADS) keys[i] = -1;
    }
    // true if `row` was not in the set yet (false, too, when no slot is left)
    __device__ bool insert(int32_t row) {
        unsigned h = slot(row);
        for (int probe = 0; probe < 1 << bits; ++probe, h = next(h)) {
            const int32_t old = atomicCAS(&keys[h], -1, row);
            if (old == -1) return true;
            if (old == row) return false;
        }
        return false;
    }
};
int set_bits(int limit) {
    int b = 6;
    while (1 << b < 2 * limit) ++b;
    return b;
}
size_t rings_lds(int limit) { return ((size_t)4 << set_bits(limit)) + 2 * (size_t)limit * 4 + 16; }

// Rings of the tile [r0, r1): counts to ring[0 .. CHAIN_MAX_STEPS] (-1 from the ring on with which
// the halo exceeds `limit` rows), halo rows, ascending inside a ring, to ext (null: counts only).
__device__ void collect_rings(const ChainMatrix& m, int64_t r0, int64_t r1, int max_steps, int limit, int bits,
                              char* smem, int32_t* ring, int32_t* ext) {
    RowSet set{reinterpret_cast<int32_t*>(smem), bits};
    int32_t* fresh = set.keys + (1 << bits);  // the ring being collected
    int32_t* last = fresh + limit;            // the ring before
    int& shared_count = *(last + limit);
    const int t = threadIdx.x;
    set.clear();
    int total = 0, front = (int)(r1 - r0);  // halo rows so far; rows of the last ring
    if (t == 0) ring[0] = front;
    bool own = true, fits = true;
    for (int j = 1; j <= CHAIN_MAX_STEPS; ++j) {
        if (!fits || j > max_steps) {
            if (t == 0) ring[j] = -1;
            continue;
        }
        __syncthreads();
        if (t == 0) shared_count = 0;
        __syncthreads();
        for (int i = t; i < front; i += PLAN_THREADS) {
            int64_t row = own ? r0 + i : last[i];
            if (m.perm) row = m.perm[row];
            const int64_t sl = row >> 6, base = m.slice_ptr[sl] + (row & 63);
            for (int k = 0; k < m.slice_width[sl]; ++k) {
                int32_t c = m.indices[base + (int64_t)k * 64];
                if (m.place) c = m.place[c];
                if (c >= r0 && c < r1) continue;
                // too many already: the ring is dropped
                if (__hip_atomic_load(&shared_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) + total > limit) break;
                if (set.insert(c)) {
                    const int p = atomicAdd(&shared_count, 1);
                    if (p < limit) fresh[p] = c;
                }
            }
        }
        __syncthreads();
        const int count = shared_count;
        if (total + count > limit) {
            fits = false;
            if (t == 0) ring[j] = -1;
            continue;
        }
        if (ext) {  // ascending: any insertion order gives the same plan
            for (int i = t; i < count; i += PLAN_THREADS) {
                const int32_t row = fresh[i];
                int rank = 0;
                for (int q = 0; q < count; ++q) rank += fresh[q] < row;
                last[rank] = row;
                ext[total + rank] = row;
            }
        } else {
            int32_t* swap = fresh;
            fresh = last;
            last = swap;
        }
        total += count;
        front = count;
        own = false;
        if (t == 0) ring[j] = (int)(r1 - r0) + total;
    }
}

struct SampleArgs {
    int heights[CHAIN_CANDIDATES];
    int capacity, bits;
};

__global__ __launch_bounds__(PLAN_THREADS) void k_chain_sample(ChainMatrix m, SampleArgs h, int32_t* out) {
    extern __shared__ __align__(16) char smem[];
    const int c = blockIdx.x / CHAIN_SAMPLES, s = blockIdx.x % CHAIN_SAMPLES;
    const int64_t rows = h.heights[c], ntiles = (m.n + rows - 1) / rows;
    const int64_t t = ntiles <= CHAIN_SAMPLES ? (s < ntiles ? s : ntiles - 1) : s * ntiles / CHAIN_SAMPLES;
    const int64_t r0 = t * rows, r1 = r0 + rows < m.n ? r0 + rows : m.n;
    collect_rings(m, r0, r1, CHAIN_MAX_STEPS, min(CHAIN_MAX_HALO, h.capacity - (int)rows), h.bits, smem,
                  out + (int64_t)blockIdx.x * (CHAIN_MAX_STEPS + 1), nullptr);
}

__global__ __launch_bounds__(PLAN_THREADS) void k_chain_rings(ChainMatrix m, const int32_t* tile_begin, int max_steps,
                                                              int bits, int32_t* ring, int32_t* ext, int64_t ext_stride) {
    extern __shared__ __align__(16) char smem[];
    const int64_t t = blockIdx.x;
    collect_rings(m, tile_begin[t], tile_begin[t + 1], max_steps, (int)ext_stride, bits, smem,
                  ring + t * (CHAIN_MAX_STEPS + 1), ext + t * ext_stride);
}

__device__ __forceinline__ bool is_zero(float v) { return v == 0.f; }
__device__ __forceinline__ bool is_zero(double v) { return v == 0.0; }
template <class R> __device__ __forceinline__ bool is_zero(cplx<R> v) { return v.re == R(0) && v.im == R(0); }

// Entries of every local row up to distance steps - 1: 2-byte local columns (a missing entry is the
// zero row), codes or values, and the diagonal.
template <class V, int FORM>
__global__ __launch_bounds__(PLAN_THREADS) void k_chain_entries(ChainMatrix m, const int32_t* tile_begin,
                                                                const int32_t* ring, const int32_t* ext,
                                                                int64_t ext_stride, int bits, int steps, int groups,
                                                                int zero_item, int ew,
                                                                int rows_y, ushort4* lidx, uint32_t* codes, V* vals,
                                                                V* diag) {
    extern __shared__ __align__(16) char smem[];
    RowSet set{reinterpret_cast<int32_t*>(smem), bits};
    int32_t* keys = set.keys;
    uint16_t* place = reinterpret_cast<uint16_t*>(keys + (1 << bits));
    const int64_t t = blockIdx.x;
    const int64_t r0 = tile_begin[t];
    const int own = (int)(tile_begin[t + 1] - r0);
    const int32_t* rg = ring + t * (CHAIN_MAX_STEPS + 1);
    const int32_t* halo = ext + t * ext_stride;
    const int nx = rg[steps], ny = rg[steps - 1];
    set.clear();
    __syncthreads();
    for (int i = threadIdx.x; i < nx - own; i += PLAN_THREADS) {
        const int32_t row = halo[i];
        unsigned h = set.slot(row);
        while (atomicCAS(&keys[h], -1, row) != -1) h = set.next(h);  // fewer rows than slots
        place[h] = (uint16_t)((own + i) * ew);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < rows_y; i += PLAN_THREADS) {
        // rows past the tile's last are padding: no entries
        int64_t row = i < own ? r0 + i : i < ny ? halo[i - own] : r0;
        if (m.perm) row = m.perm[row];
        const int64_t sl = row >> 6, base = m.slice_ptr[sl] + (row & 63);
        // local column of a neighbour (every one lies within `steps` of the tile)
        auto local = [&](int32_t col) -> uint16_t {
            if (m.place) col = m.place[col];
            if (col >= r0 && col < r0 + own) return (uint16_t)((col - r0) * ew);
            unsigned h = set.slot(col);
            while (keys[h] != col && keys[h] != -1) h = set.next(h);
            return keys[h] == col ? place[h] : (uint16_t)zero_item;
        };
        const bool ordered = FORM != CHAIN_STD && m.ordered();
        const int w = i >= ny ? 0 : ordered ? m.row_width[sl] : m.slice_width[sl];
        int next = 0;  // ordered: the next off-diagonal entry
        for (int g = 0; g < groups; ++g) {
            uint16_t id[4];
            uint32_t code = 0;
            for (int q = 0; q < 4; ++q) {
                const int k = 4 * g + q;
                id[q] = (uint16_t)zero_item;
                V v = zero(V{});
                if (k < w) {
                    if constexpr (FORM == CHAIN_STD) {
                        const int64_t e = base + (int64_t)k * 64;
                        v = static_cast<const V*>(m.vals)[e];
                        id[q] = local(m.indices[e]);
                    } else if (ordered) {
                        const int64_t e = m.row_ptr[sl] + (row & 63) + (int64_t)k * 64;
                        const int32_t col = m.row_indices[e];
                        if (col != row) {
                            const uint32_t cd = m.codes[base + (int64_t)next * 64];
                            ++next;
                            code |= cd << (8 * q);
                            if (!(FORM == CHAIN_UNIFORM && cd == 0)) id[q] = local(col);
                        } else if (!is_zero(static_cast<const V*>(m.row_vals)[e])) {
                            id[q] = (uint16_t)(i * ew);  // the diagonal (a padded slot is zero)
                        }
                    } else {
                        const int64_t e = base + (int64_t)k * 64;
                        const int32_t col = m.indices[e];
                        const uint32_t cd = m.codes[e];
                        if (col != row && !(FORM == CHAIN_UNIFORM && cd == 0)) {
                            code |= cd << (8 * q);
                            id[q] = local(col);
                        }
                    }
                }
                if constexpr (FORM == CHAIN_STD) vals[(t * (4 * groups) + k) * rows_y + i] = v;
            }
            lidx[(t * groups + g) * rows_y + i] = make_ushort4(id[0], id[1], id[2], id[3]);
            if constexpr (FORM == CHAIN_TABLE) codes[(t * groups + g) * rows_y + i] = code;
        }
        if constexpr (FORM != CHAIN_STD) diag[t * rows_y + i] = i < ny ? static_cast<const V*>(m.diag)[row] : zero(V{});
    }
}

// Sums over the tiles of each system, tiles in order inside 32 interleaved groups.
__global__ __launch_bounds__(1024) void k_chain_reduce(const double* partials, int64_t ntiles, int width, int cols,
                                                       const int32_t* system_tiles, int64_t num_systems, int ncol,
                                                       int kinds, int vw, int c0, double* sums) {
    __shared__ double red[1024];
    const int64_t step = blockIdx.x / num_systems, sys = blockIdx.x % num_systems;
    const int64_t t0 = system_tiles ? system_tiles[sys] : 0, t1 = system_tiles ? system_tiles[sys + 1] : ntiles;
    const int ng = 1024 / width, w = threadIdx.x % width, g = threadIdx.x / width;
    double v = 0;
    if (g < ng)
        for (int64_t t = t0 + g; t < t1; t += ng) v += partials[(step * ntiles + t) * width + w];
    red[threadIdx.x] = v;
    __syncthreads();
    if (g == 0) {
        for (int q = 1; q < ng; ++q) v += red[q * width + w];
        // item layout [kind][column of the element][element] -> [kind][column]
        const int ew = cols / ncol, e = w % ew, kc = w / ew, kind = kc / ncol, col = e * ncol + kc % ncol;
        const int slot = kind == 0 || kinds == 4 ? kind : kind + 1;
        double* o = sums + (step * num_systems + sys) * 4 * vw + c0;
        o[slot * vw + col] = v;
        if (kind == 0 && kinds < 4) o[vw + col] = 0.0;
        if (kind == 1 && kinds == 2) o[3 * vw + col] = 0.0;
    }
}

// Operator entries on the own rows of every tile (see k_chain_entries): local columns and values.
template <class V>
__global__ __launch_bounds__(PLAN_THREADS) void k_chain_op(ChainMatrix m, const int32_t* tile_begin, const int32_t* ring,
                                                           const int32_t* ext, int64_t ext_stride, int bits, int zero_item,
                                                           int ew, ChainOp o, int32_t* missing) {
    extern __shared__ __align__(16) char smem[];
    RowSet set{reinterpret_cast<int32_t*>(smem), bits};
    uint16_t* place = reinterpret_cast<uint16_t*>(set.keys + (1 << bits));
    const int64_t t = blockIdx.x, r0 = tile_begin[t];
    const int own = (int)(tile_begin[t + 1] - r0);
    const int32_t* halo = ext + t * ext_stride;
    const int near = ring[t * (CHAIN_MAX_STEPS + 1) + 1];  // rows that hold r_k at every step
    set.clear();
    __syncthreads();
    for (int i = threadIdx.x; i < near - own; i += PLAN_THREADS) {
        unsigned h = set.slot(halo[i]);
        while (atomicCAS(&set.keys[h], -1, halo[i]) != -1) h = set.next(h);  // fewer rows than slots
        place[h] = (uint16_t)((own + i) * ew);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < o.rows; i += PLAN_THREADS) {
        const int64_t row = i < own ? r0 + i : r0;
        const int64_t sl = row >> 6, base = m.slice_ptr[sl] + (row & 63);
        const int w = i < own ? m.slice_width[sl] : 0;
        for (int g = 0; g < o.groups; ++g) {
            uint16_t id[4];
            for (int q = 0; q < 4; ++q) {
                const int k = 4 * g + q;
                id[q] = (uint16_t)zero_item;
                V v = zero(V{});
                if (k < w) {
                    const int32_t c = m.indices[base + (int64_t)k * 64];
                    v = static_cast<const V*>(m.vals)[base + (int64_t)k * 64];
                    if (c >= r0 && c < r0 + own) {
                        id[q] = (uint16_t)((c - r0) * ew);
                    } else {
                        unsigned h = set.slot(c);
                        while (set.keys[h] != c && set.keys[h] != -1) h = set.next(h);
                        if (set.keys[h] == c) id[q] = place[h];
                        else *missing = 1;
                    }
                }
                static_cast<V*>(o.vals)[(t * (4 * o.groups) + k) * o.rows + i] = v;
            }
            o.lidx[(t * o.groups + g) * o.rows + i] = make_ushort4(id[0], id[1], id[2], id[3]);
        }
    }
}

// most LDS of a plan kernel: a set of CHAIN_MAX_HALO rows and two rings
const size_t PLAN_LDS = rings_lds(CHAIN_MAX_HALO);

}  // namespace

template <class F>
static int with_shape(int scalar, int cols, int form, int width, F&& f) {
    return with_layout(scalar, cols, [&](auto e, auto ew) {
        auto of = [&](auto form_) {
            using E = decltype(e);
            constexpr int EW = decltype(ew)::value, F_ = decltype(form_)::value;
            return width <= 4 ? f(shape<E, EW, F_, true>{}, ew) : f(shape<E, EW, F_, false>{}, ew);
        };
        if (form == CHAIN_STD) return of(std::integral_constant<int, CHAIN_STD>{});
        if (form == CHAIN_TABLE) return of(std::integral_constant<int, CHAIN_TABLE>{});
        return of(std::integral_constant<int, CHAIN_UNIFORM>{});
    });
}

int chain_max_cols(int scalar) { return scalar == 0 ? 16 : scalar == 3 ? 4 : 8; }

int chain_row_capacity(const ChainMatrix& m, int cols) {
    if (m.adjoint) return chain_adjoint_capacity(m.scalar, cols);
    return with_shape(m.scalar, cols, m.form(), m.width(), [](auto s, auto) { return decltype(s)::rows; });
}

int chain_row_items(int scalar, int cols) {
    return with_layout(scalar, cols, [](auto, auto ew) { return decltype(ew)::value; });
}

int chain_row_pad(const ChainMatrix& m, int cols) {
    if (m.adjoint) return chain_adjoint_row_pad(m.scalar, cols);
    return with_shape(m.scalar, cols, m.form(), m.width(),
                      [](auto s, auto ew) { return decltype(s)::threads / decltype(ew)::value; });
}

int chain_partial_width(int scalar, int cols, int mode) {
    if (mode == CHAIN_DOTS) return scalar >= 2 ? 4 : 2;
    return with_shape(scalar, cols, CHAIN_STD, 1, [](auto s, auto ew) { return decltype(s)::NS * decltype(ew)::value; });
}

int launch_chain(const ChainLaunch& L, hipStream_t s) {
    if (!L.plan || L.steps < 1 || L.steps > L.plan->steps || L.plan->rows_x > chain_row_capacity(L.m, L.cols) ||
        L.col_groups < 1 || (L.col_groups > 1 && L.mode != CHAIN_SUMS))
        return -1;
    switch (L.m.scalar) {
        case 0: return launch_chain_f32(L, s);
        case 1: return launch_chain_f64(L, s);
        case 2: return launch_chain_c64(L, s);
        default: return launch_chain_c128(L, s);
    }
}

void launch_chain_reduce(int scalar, int mode, const double* partials, int64_t ntiles, int cols, int64_t nsteps,
                         const int32_t* system_tiles, int64_t num_systems, int vw, int c0, double* sums, hipStream_t s) {
    const int width = chain_partial_width(scalar, cols, mode);
    const int ncol = with_layout(scalar, cols, [](auto e, auto) { return elem<decltype(e)>::cols; });
    hipLaunchKernelGGL(k_chain_reduce, dim3((unsigned)(nsteps * num_systems)), dim3(1024), 0, s, partials, ntiles, width,
                       cols, system_tiles, num_systems, ncol, width / cols, vw, c0, sums);
}

int chain_sample(const ChainMatrix& m, const int* heights, int count, int capacity, int32_t* out, hipStream_t s) {
    SampleArgs h{};
    int limit = 1;
    for (int i = 0; i < count; ++i) {
        h.heights[i] = heights[i];
        limit = std::max(limit, std::min(CHAIN_MAX_HALO, capacity - heights[i]));
    }
    h.capacity = capacity;
    h.bits = set_bits(limit);
    const size_t bytes = rings_lds(limit);
    static std::atomic<uint64_t> allowed{0};
    if (!allow_lds(reinterpret_cast<const void*>(k_chain_sample), PLAN_LDS, allowed)) return -1;
    hipLaunchKernelGGL(k_chain_sample, dim3(count * CHAIN_SAMPLES), dim3(PLAN_THREADS), bytes, s, m, h, out);
    return 0;
}

int chain_rings(const ChainMatrix& m, const ChainPlan& P, int max_steps, hipStream_t s) {
    const size_t bytes = rings_lds((int)P.ext_stride);
    static std::atomic<uint64_t> allowed{0};
    if (!allow_lds(reinterpret_cast<const void*>(k_chain_rings), PLAN_LDS, allowed)) return -1;
    hipLaunchKernelGGL(k_chain_rings, dim3((unsigned)P.ntiles), dim3(PLAN_THREADS), bytes, s, m, P.tile_begin, max_steps,
                       set_bits((int)P.ext_stride), P.ring, P.ext, P.ext_stride);
    return 0;
}

template <class V, int FORM>
static int entries_of(const ChainMatrix& m, const ChainPlan& P, hipStream_t s) {
    auto kernel = k_chain_entries<V, FORM>;
    const int bits = set_bits(std::max<int>(1, (int)P.ext_stride));
    const size_t bytes = ((size_t)1 << bits) * (sizeof(int32_t) + sizeof(uint16_t));
    static std::atomic<uint64_t> allowed{0};
    if (!allow_lds(reinterpret_cast<const void*>(kernel), PLAN_LDS, allowed)) return -1;
    hipLaunchKernelGGL(kernel, dim3((unsigned)P.ntiles), dim3(PLAN_THREADS), bytes, s, m, P.tile_begin, P.ring, P.ext,
                       P.ext_stride, bits, P.steps, P.groups, P.rows_x * P.row_items, P.row_items, P.rows_y, P.lidx,
                       P.codes, static_cast<V*>(P.vals), static_cast<V*>(P.diag));
    return 0;
}

int chain_entries(const ChainMatrix& m, const ChainPlan& P, hipStream_t s) {
    auto by_form = [&](auto v) {
        using V = decltype(v);
        switch (m.form()) {
            case CHAIN_STD: return entries_of<V, CHAIN_STD>(m, P, s);
            case CHAIN_TABLE: return entries_of<V, CHAIN_TABLE>(m, P, s);
            default: return entries_of<V, CHAIN_UNIFORM>(m, P, s);
        }
    };
    switch (m.scalar) {
        case 0: return by_form(float{});
        case 1: return by_form(double{});
        case 2: return by_form(cf32{});
        default: return by_form(cf64{});
    }
}

template <class V>
static int op_entries_of(const ChainMatrix& op, const ChainPlan& P, const ChainOp& o, int32_t* missing, hipStream_t s) {
    auto kernel = k_chain_op<V>;
    const int bits = set_bits(std::max<int>(1, (int)P.ext_stride));
    const size_t bytes = ((size_t)1 << bits) * (sizeof(int32_t) + sizeof(uint16_t));
    static std::atomic<uint64_t> allowed{0};
    if (!allow_lds(reinterpret_cast<const void*>(kernel), PLAN_LDS, allowed)) return -1;
    hipLaunchKernelGGL(kernel, dim3((unsigned)P.ntiles), dim3(PLAN_THREADS), bytes, s, op, P.tile_begin, P.ring, P.ext,
                       P.ext_stride, bits, P.rows_x * P.row_items, P.row_items, o, missing);
    return 0;
}

int chain_op_entries(const ChainMatrix& op, const ChainPlan& P, const ChainOp& o, int32_t* missing, hipStream_t s) {
    switch (op.scalar) {
        case 0: return op_entries_of<float>(op, P, o, missing, s);
        case 1: return op_entries_of<double>(op, P, o, missing, s);
        case 2: return op_entries_of<cf32>(op, P, o, missing, s);
        default: return op_entries_of<cf64>(op, P, o, missing, s);
    }
}

}  // namespace kpmx
