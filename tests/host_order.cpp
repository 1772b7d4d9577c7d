// The host core's matrix in a given site order against the plain way: scaled in the original order, then
// rows and columns permuted and every row sorted.  Prints the number of differing matrices.
#include "../pybinding_amd/csrc/core/kpm_core.hpp"

#include <cstdio>
#include <random>

using namespace kpmx_host;

template <class T>
int differs(int n, int width, double missing_diagonal, Scale<> scale, unsigned seed) {
    std::mt19937 rng(seed);
    std::uniform_real_distribution<double> real(-1, 1);
    Csr<T> h;
    h.rows = h.cols = n;
    h.indptr.push_back(0);
    for (int r = 0; r < n; ++r) {
        std::vector<int32_t> cols;
        const int w = (int)(rng() % (unsigned)(width + 1));
        for (int k = 0; k < w; ++k) cols.push_back((int32_t)(rng() % (unsigned)n));
        if (0.5 * (real(rng) + 1) >= missing_diagonal) cols.push_back(r);
        std::sort(cols.begin(), cols.end());
        cols.erase(std::unique(cols.begin(), cols.end()), cols.end());
        for (auto c : cols) {
            h.indices.push_back(c);
            h.data.push_back(T(real(rng)));
        }
        h.indptr.push_back((int32_t)h.indices.size());
    }
    std::vector<int32_t> order((size_t)n);
    for (int i = 0; i < n; ++i) order[(size_t)i] = i;
    std::shuffle(order.begin(), order.end(), rng);

    const Indices sites(n / 2, std::vector<idx_t>{0, n - 1});
    OptimizedHamiltonian<T> ordered(&h, true), plain(&h, false);
    ordered.locality_order = order;
    ordered.optimize_for(sites, scale, true);
    plain.optimize_for(sites, scale);
    plain.reorder_map = order;
    const Csr<T> ref = plain.reorder(plain.h2);
    bool same = ordered.h2.indptr == ref.indptr && ordered.h2.indices == ref.indices && ordered.h2.data == ref.data &&
                ordered.h2.rows == n && ordered.h2.cols == n && ordered.reorder_map == order;
    same = same && ordered.optimized_idx.src[0] == order[(size_t)(n / 2)] && ordered.optimized_idx.dest[1] == order[(size_t)(n - 1)];
    return same ? 0 : 1;
}

int main() {
    int bad = 0;
    for (unsigned seed = 0; seed < 4; ++seed)
        for (int n : {1, 2, 5, 64, 777})
            for (int width : {0, 1, 3, 4, 5, 19})
                for (double missing : {0.0, 0.5, 1.0})
                    for (auto scale : {Scale<>(-9, 9), Scale<>(-3, 6)}) {
                        bad += differs<double>(n, width, missing, scale, seed);
                        bad += differs<float>(n, width, missing, scale, seed);
                        bad += differs<std::complex<double>>(n, width, missing, scale, seed);
                    }
    std::printf("%d\n", bad);
    return bad != 0;
}
