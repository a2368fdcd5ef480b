// Host-side rules of libs4f's launch sequences, on the CPU: every check named
// on the command line, or all.  Prints the failing ones.
#include "../solids4foam_amd/csrc/s4f_api.hip"
using namespace s4f;

static int failures = 0;
#define CHECK(x) \
    do { \
        if (!(x)) { \
            ++failures; \
            std::printf("%s:%d: %s\n", __func__, __LINE__, #x); \
        } \
    } while (0)

// control block at a look: iCorr outer iterations done with pcg PCG iterations in all
static Ctl ctlAt(int iCorr, long long pcg, int n = 0) {
    Ctl c;
    std::memset(&c, 0, sizeof(c));
    c.iCorr = iCorr;
    c.pcgTotal = pcg;
    c.nIter[0] = n;
    return c;
}

// PCG iterations of a pass after looks at instances of steady counts
static int passLength(bool mg, const std::vector<double>& perOuter) {
    PassRule rule(perOuter.size());
    std::vector<int> live;
    for (int i = 0; i < (int)perOuter.size(); ++i) {
        for (int it = 10; it <= 200; it += 10) rule.look(i, ctlAt(it, (long long)(it * perOuter[i])));
        live.push_back(i);
    }
    return rule.choose(mg, live, 1000);
}

static void passRule() {
    // a steady count: one pass per outer iteration, nothing empty
    for (int u : {1, 2, 3, 4, 5, 6, 8}) CHECK(passLength(true, {(double)u}) == u);
    CHECK(passLength(true, {1.1}) == 1);      // the odd second iteration in a pass of its own
    CHECK(passLength(true, {3.6}) == 4);
    CHECK(passLength(true, {0.0}) == 1);      // no PCG iteration needed
    // (1/2 + k) times the passes of all: 4.5 x 7 against 2.5 x 13, and 4.5 x 4 against 2.5 x 7
    CHECK(passLength(true, {4, 4, 4, 4, 4, 4, 1}) == 4);
    CHECK(passLength(true, {4, 4, 4, 1}) == 2);
    CHECK(passLength(true, {1, 1, 1, 1, 1, 1, 1, 2}) == 1);
    // long diagonal solves: passes of many iterations
    for (double u : {90.0, 95.0, 97.0, 216.0}) CHECK(passLength(false, {u}) >= 12);
    // a first outer iteration longer than a look counts as what it has used so far
    PassRule rule(1);
    rule.look(0, ctlAt(0, 0, 40));
    CHECK(rule.choose(false, {0}, 1000) >= 8);
    rule.reset(0);
    CHECK(rule.choose(true, {0}, 1000) == 1);
    // a short solve takes short passes
    rule.look(0, ctlAt(4, 24));
    CHECK(rule.choose(true, {0}, 1) == 2 && rule.choose(true, {0}, 24) == 3 && rule.choose(true, {0}, 48) == 6);
    // the instance with most of the iterations left decides
    auto at = [](int iCorr, long long pcg, double res) {
        Ctl c = ctlAt(iCorr, pcg);
        c.solTol = c.altTol = 1e-8;
        c.nCorr = 100000;
        c.initResMag = res;
        return c;
    };
    PassRule two(3);
    for (int i = 0; i < 2; ++i) two.look(i, at(100, 200, 1e-7));
    two.look(2, at(100, 105, 0.4));
    CHECK(two.choose(true, {0, 1, 2}, 1000) == 1);
    two.look(2, at(100, 105, 2e-8));
    CHECK(two.choose(true, {0, 1, 2}, 1000) == 2);
    two.look(2, at(100, 105, NAN));
    CHECK(two.choose(true, {0, 1, 2}, 1000) == 2);
}

static void progressWatch() {
    ProgressWatch watch(2);
    auto looks = [&](int i, Ctl c, int n) {
        try {
            for (int k = 0; k < n; ++k) watch.look(i, c);
        } catch (const HipError&) {
            return true;
        }
        return false;
    };
    Ctl c = ctlAt(0, 0);
    for (int k = 0; k < 200; ++k) {  // steps of a PCG, of an outer loop without one
        ++c.pIt;
        CHECK(!looks(0, c, 1));
    }
    for (int k = 0; k < 200; ++k) {
        ++c.iCorr;
        CHECK(!looks(0, c, 1));
        CHECK(!looks(1, c, 1));
    }
    c.pending = 99;  // a step that no launch takes on; the other instance goes on
    CHECK(!looks(0, c, 4));
    ++c.iCorr;
    CHECK(!looks(1, c, 4));
    CHECK(!looks(0, c, 4));
    CHECK(looks(0, c, 100));
    CHECK(!looks(1, c, 2));
}

static void lduSlots() {
    CHECK(lduSlotCount(6, 100, 600) == 6);
    CHECK(lduSlotCount(6, 100, 480) == 6);  // a quarter more entries
    CHECK(lduSlotCount(6, 100, 479) == 0);
    CHECK(lduSlotCount(4, 100, 320) == 4);
    CHECK(lduSlotCount(5, 100, 500) == 6);
    CHECK(lduSlotCount(7, 100, 700) == 0);
    CHECK(lduSlotCount(0, 1, 0) == 0);      // a single cell
    // rows of five: their entries can be numbered, six for each could not
    const int most = INT32_MAX / (6 * kSlice);
    CHECK(lduSlotCount(5, most, 5LL * most) == 6);
    CHECK(lduSlotCount(5, most + 1, 5LL * (most + 1)) == 0);
}

int main(int argc, char** argv) {
    const std::string only = argc > 1 ? argv[1] : "";
    const std::pair<const char*, void (*)()> checks[] = {{"passRule", passRule}, {"progressWatch", progressWatch},
                                                         {"lduSlots", lduSlots}};
    for (const auto& c : checks)
        if (only.empty() || only == c.first) c.second();
    return failures ? 1 : 0;
}
