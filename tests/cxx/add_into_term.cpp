// mrcpp::add of a FunctionTreeVector into one of its own terms: accepted for any but the last of
// three or more terms, refused otherwise, with the result of a sum into another tree.
#include <cmath>
#include <cstdio>

#include "mwg_mrcpp.hpp"

int main() {
    const int corner[3] = {-1, -1, -1}, boxes[3] = {2, 2, 2};
    mrcpp::BoundingBox<3> world(-4, corner, boxes);
    mrcpp::LegendreBasis basis(5);
    mrcpp::MultiResolutionAnalysis<3> MRA(world, basis, 12);
    int fails = 0;
    const double prec = 1e-4;
    mrcpp::FunctionTree<3> f0(MRA), f1(MRA), f2(MRA);
    mrcpp::FunctionTree<3> *f[3] = {&f0, &f1, &f2};
    for (int i = 0; i < 3; i++) {
        mrcpp::GaussExp<3> e;
        e.append(mrcpp::GaussFunc<3>(3.0 + 4.0 * i, 1.0, {0.3 * i, -0.2, 0.5 - 0.4 * i}));
        mrcpp::project(prec, *f[i], e);
    }
    const double c[3] = {0.7, -1.3, 2.0};
    mrcpp::FunctionTree<3> ref(MRA), diff(MRA);
    mrcpp::FunctionTreeVector<3> terms{{c[0], &f0}, {c[1], &f1}, {c[2], &f2}};
    mrcpp::add(prec, ref, terms);
    for (int own = 0; own < 3; own++) {
        mrcpp::FunctionTree<3> out(MRA);
        mrcpp::copy_func(out, *f[own]);
        terms[own] = std::make_tuple(c[own], &out);
        bool thrown = false;
        try {
            mrcpp::add(prec, out, terms);
        } catch (const mrcpp::Error &e) {
            thrown = true;
            std::printf("out = term %d: %s\n", own, e.what());
        }
        terms[own] = std::make_tuple(c[own], f[own]);
        bool ok = thrown == (own == 2);
        if (!thrown) {
            mrcpp::add(prec, diff, 1.0, out, -1.0, ref);
            ok = ok && out.getNNodes() == ref.getNNodes() && diff.getSquareNorm() == 0.0;
        }
        std::printf("%s: out = term %d of 3\n", ok ? "ok" : "FAILED", own);
        fails += ok ? 0 : 1;
    }
    for (int own = 0; own < 2; own++) {
        mrcpp::FunctionTreeVector<3> two{{c[0], &f0}, {c[1], &f1}};
        bool thrown = false;
        try {
            mrcpp::add(prec, *f[own], two);
        } catch (const mrcpp::Error &) {
            thrown = true;
        }
        std::printf("%s: out = term %d of 2 is refused\n", thrown ? "ok" : "FAILED", own);
        fails += thrown ? 0 : 1;
    }
    std::printf("%s\n", fails ? "add into a term: FAILED" : "add into a term: ok");
    return fails ? 1 : 0;
}
