// Which form of the projection GEMM a launch takes (csrc/linear_forms.h), for tests that mean a certain one: index into the table of its
// kind. mnk: rows, output features and contraction of each of the n problems.
#include "linear_forms.h"

extern "C" int linear_form(const int* mnk, int n, int int8_weights, int geglu, int compute_units) {
    static const float scale = 1.f;
    mi::LinearBatch b{};
    for (int i = 0; i < n; ++i) {
        b.p[i].M = mnk[3 * i];
        b.p[i].N = mnk[3 * i + 1];
        b.p[i].K = mnk[3 * i + 2];
        b.p[i].w_scale = int8_weights ? &scale : nullptr;
    }
    return mi::gemm::pick_form(b, n, geglu != 0, compute_units);
}
