// Host-only check of the settling plans: over random networks and batches, no
// problem of any step has split-K partial tiles or counters outside the scratch
// its workspace holds, in the allocation-free variant's layout (drawn towards
// the end of its array) and in the allocating one's.  Nothing here touches a
// GPU; pointers are offsets from a made-up base that is never read.
//   plan_check SEED COUNT                    random plans
//   plan_check DTYPE BATCH SIZE SIZE ...     one plan
#include "../../predicitivecoding_amd/csrc/pcdevice.hip"

#include <cstdio>
#include <cstdlib>
#include <random>

static char* const kBase = (char*)((size_t)1 << 40);

static void set_net(pcd_model* m, const std::vector<int>& sizes, int dtype) {
    m->L = (int)sizes.size();
    m->s = sizes;
    m->P.resize(m->L);
    for (int l = 0; l < m->L; ++l) m->P[l] = (int)round_up(sizes[l], kFeatPad);
    m->dtype = dtype;
    m->W.assign(m->L, nullptr);
    m->WT = m->Wpk = m->WTpk = m->W;
    m->bias.assign(m->L, nullptr);
    m->prec.assign(m->L, 1.f);
    if (!direct_eligible(m)) m->Wpk.clear(), m->WTpk.clear();
    else for (int l = 1; l < m->L; ++l) m->Wpk[l] = m->WTpk[l] = kBase;
}

// The furthest byte past `w`'s split scratch that the step loop's problems
// reach (0: none); *shares is set when steps with one-row layers ran.
static size_t beyond(const pcd_model* m, const Workspace& w, int batch, Tile tile, size_t part_end, size_t count_end,
                     bool* shares) {
    size_t over = 0;
    std::vector<ProblemSet> err, upd;
    int nslots = 0, shared_from = 0;
    auto look = [&]() {
        for (const auto* sets : {&err, &upd})
            for (const ProblemSet& ps : *sets)
                for (int i = 0; i < ps.n; ++i) {
                    const Problem& p = ps.p[i];
                    if (p.ksplit <= 1) continue;
                    const size_t pe = (size_t)(p.part + (size_t)p.tiles * tile.m * tile.n);
                    const size_t ce = (size_t)(p.count + p.tiles / p.ksplit);
                    if (pe > part_end) over = std::max(over, pe - part_end);
                    if (ce > count_end) over = std::max(over, ce - count_end);
                }
    };
    build_phase_sets(m, &w, batch, tile, 0, err, upd, &nslots);
    look();
    RelaxSpec r;
    r.batch = batch;
    r.steps = m->L;
    r.tile = tile;
    *shares = use_front(m, &w, r);
    for (int t = 0; *shares && t < m->L - 1; ++t) {
        build_front_sets(m, &w, batch, tile, t, err, upd, &nslots, &shared_from);
        look();
    }
    return over;
}

static int check(const pcd_model* m, int batch, bool verbose, int* accepted, int* sharing) {
    Workspace w;
    Tile tile;
    bool shares = false;
    const size_t need = plan_noalloc(m, kBase, batch, &tile, w);
    int bad = 0;
    if (need <= kNoAllocScratchBytes) {
        const size_t over = beyond(m, w, batch, tile, (size_t)kBase + need, (size_t)w.split_part, &shares);
        ++*accepted;
        *sharing += shares;
        bad += over > 0;
        if (over || verbose) {
            std::printf("%s noalloc: dtype %d rows %d tile %d need %zu over %zu shares %d:", over ? "BAD" : "ok", m->dtype,
                        batch, tile.m, need, over, (int)shares);
            for (int v : m->s) std::printf(" %d", v);
            std::printf("\n");
        }
    }
    // the allocating variant: as ensure_workspace sizes the scratch
    Workspace a;
    tile = choose_tile(m, batch);
    carve_workspace(m, kBase, batch, tile, true, a);
    a.split_part = (float*)kBase;
    a.split_count = (int*)(kBase + ((size_t)1 << 36));
    const size_t over = beyond(m, a, batch, tile, (size_t)kBase + (size_t)split_part_tiles(m) * 128 * 128 * 4,
                               (size_t)a.split_count + split_count_bytes(m), &shares);
    if (over) {
        std::printf("BAD workspace: dtype %d rows %d over %zu:", m->dtype, batch, over);
        for (int v : m->s) std::printf(" %d", v);
        std::printf("\n");
    }
    return bad + (over > 0);
}

int main(int argc, char** argv) {
    int bad = 0, accepted = 0, sharing = 0;
    if (argc > 3) {
        pcd_model m;
        std::vector<int> sizes;
        for (int i = 3; i < argc; ++i) sizes.push_back(std::atoi(argv[i]));
        set_net(&m, sizes, std::atoi(argv[1]));
        std::printf("tile %d\n", choose_tile(&m, std::atoi(argv[2])).m);
        bad = check(&m, std::atoi(argv[2]), true, &accepted, &sharing);
    } else {
        std::mt19937 rng((unsigned)std::atoi(argv[1]));
        auto uniform = [&](int lo, int hi) { return std::uniform_int_distribution<int>(lo, hi)(rng); };
        auto log_uniform = [&](double lo, double hi) {
            return (int)std::exp(std::uniform_real_distribution<double>(std::log(lo), std::log(hi))(rng));
        };
        for (int i = 0; i < std::atoi(argv[2]); ++i) {
            pcd_model m;
            std::vector<int> sizes(uniform(2, 9));
            const bool equal = uniform(0, 1);
            const int width = log_uniform(16, 9000);
            for (int& v : sizes) v = equal ? width : log_uniform(8, 9000);
            set_net(&m, sizes, uniform(0, 2));
            // the largest batch that the array takes, and batches below it
            int lo = 1, hi = 1 << 20;
            Workspace w;
            Tile tile;
            while (lo + 1 < hi) {
                const int mid = lo + (hi - lo) / 2;
                (plan_noalloc(&m, kBase, mid, &tile, w) <= kNoAllocScratchBytes ? lo : hi) = mid;
            }
            for (int k = 0; k < 4; ++k)
                bad += check(&m, k == 0 ? lo : k == 1 ? std::max(1, lo - uniform(0, 64)) : log_uniform(1, lo + 1.0), false,
                             &accepted, &sharing);
        }
    }
    std::printf("%d accepted, %d with shared rows, %d bad\n", accepted, sharing, bad);
    return bad ? 1 : 0;
}
