// Simulation<...> with counting policies over an engine of stubs: prints the
// order in which policy hooks and engine calls are reached (test_policy_hooks.py).
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../pansim_amd/csrc/host/simulation.h"

struct pansim_ctx {};
static pansim_ctx g_ctx;
static std::string g_log;
static void say(const char* what) { g_log += (g_log.empty() ? "" : " ") + std::string(what); }

extern "C" {
const char* pansim_create_error(void) { return ""; }
const char* pansim_last_error(const pansim_ctx*) { return ""; }
int pansim_create(pansim_ctx** out, const pansim_dims*, const pansim_tables*, const pansim_locations*, const pansim_agents*,
                  uint64_t, uint32_t, uint32_t, uint32_t, uint32_t) {
    *out = &g_ctx;
    return 0;
}
void pansim_destroy(pansim_ctx*) {}
int pansim_movement_step(pansim_ctx*, const pansim_step_params*) { return say("move"), 0; }
int pansim_infection_step(pansim_ctx*, uint32_t, uint32_t, float, float, uint32_t) { return say("infect"), 0; }
int pansim_run_steps(pansim_ctx*, const pansim_step_params*, uint32_t n, uint32_t, float, float) {
    return say(("run" + std::to_string(n)).c_str()), 0;
}
int pansim_plan_locations(pansim_ctx*, const pansim_step_params*) { return say("plan"), 0; }
int pansim_rebuild_locations(pansim_ctx*) { return say("rebuild"), 0; }
int pansim_dummy_plan_locations(pansim_ctx*) { return 0; }
int pansim_dummy_movement_step(pansim_ctx*, uint32_t) { return 0; }
int pansim_testing_day(pansim_ctx*, uint32_t, uint32_t, const double*, uint32_t, uint32_t, uint32_t, uint32_t out[3]) {
    out[0] = out[1] = out[2] = 0;
    return say("testing"), 0;
}
int pansim_progression_day(pansim_ctx*, uint32_t, uint32_t) { return say("progression"), 0; }
int pansim_immunization_day(pansim_ctx*, uint32_t, uint32_t, const float*, const int32_t*, const float*) {
    return say("immunization"), 0;
}
int pansim_midnight_day(pansim_ctx*, pansim_midnight* m) {
    m->stats_len = 40;
    std::string s = "midnight(";
    if (m->testing) s += "t";
    if (m->progression) s += "p";
    if (m->immunization) s += "i";
    if (m->other_disease) s += "o";
    if (m->statistics) s += "s";
    return say((s + ")").c_str()), 0;
}
int pansim_vaccination_init(pansim_ctx*, const int32_t*, const float*) { return 0; }
int pansim_age_group_counts(pansim_ctx*, uint32_t out[10]) {
    for (int g = 0; g < 10; ++g) out[g] = 1;
    return 0;
}
int pansim_booster_round(pansim_ctx*, uint32_t, uint32_t, uint32_t, uint32_t, const float*) { return 0; }
int pansim_vaccinate(pansim_ctx*, uint32_t, uint32_t, uint32_t, uint32_t*, uint32_t* today) { return *today = 0, 0; }
int pansim_other_disease_day(pansim_ctx*, uint32_t, uint32_t, float) { return say("other"), 0; }
int pansim_count_hospitalized_covid(pansim_ctx*, uint32_t, uint32_t, uint32_t* out) { return *out = 0, 0; }
int pansim_count_variants(pansim_ctx*, uint32_t* out) { return out[0] = 1, 0; }
int pansim_stats_day(pansim_ctx*, uint32_t, uint32_t, const uint32_t*, uint32_t, uint32_t*, size_t, size_t* len) {
    *len = 40;
    return say("statistics"), 0;
}
int pansim_set_open_by_type(pansim_ctx*, const uint32_t*, uint32_t, uint32_t) { return 0; }
int pansim_scale_infectiousness(pansim_ctx*, double, uint32_t) { return 0; }
int pansim_expose_mutation(pansim_ctx*, uint32_t, uint32_t, double) { return 0; }
int pansim_upload_schedules(pansim_ctx*, const uint32_t*, uint32_t, const pansim_event*, uint32_t) { return 0; }
int pansim_download_field(pansim_ctx*, const char*, uint32_t, uint32_t*, size_t) { return 0; }
int pansim_infection_dump_enable(pansim_ctx*, uint32_t) { return 0; }
int pansim_infection_dump_collect(pansim_ctx*, uint32_t*, uint32_t*, size_t, size_t* a, uint32_t*, uint32_t*, float*, size_t,
                                  size_t* b) {
    return *a = *b = 0, 0;
}
}

using namespace ps;

template <class S>
struct OwnMovement : RealMovement<S> {
    void movement(Timehandler t, unsigned dt) {
        say("hook:movement");
        RealMovement<S>::movement(t, dt);
    }
};
template <class S>
struct OwnInfection : BasicInfection<S> {
    void infectionsAtLocationsMask(const Timehandler& t, unsigned dt, uint32_t mask) {
        say("hook:infection");
        BasicInfection<S>::infectionsAtLocationsMask(t, dt, mask);
    }
};
// the hooks that Simulation calls, and nothing else
template <class S>
struct MinimalInfection {
    void initializeArgs(const Options&) {}
    void finalize() {}
    void infectionsAtLocationsMask(const Timehandler&, unsigned, uint32_t) { say("hook:infection"); }
};
template <class S>
struct OwnClosure : NoClosure<S> {
    void step(Timehandler, unsigned) { say("hook:closure"); }
};
template <class S>
struct OwnTesting : DetailedTesting<S> {
    void performTests(Timehandler t, unsigned dt) {
        say("hook:testing");
        DetailedTesting<S>::performTests(t, dt);
    }
};
// a derived movement policy that changes no hook and says so
template <class S>
struct NamedMovement : RealMovement<S> {
    using EngineHooks = NamedMovement;
};

template <template <typename> class M, template <typename> class I, template <typename> class T, template <typename> class C>
static void drive(const char* name, const Options& o, unsigned n) {
    Simulation<std::array<double, 2>, unsigned, DynamicPPState, BasicAgentMeta, M, I, T, C> sim(o, false);
    if (!sim.succesfullyInitialized) {
        std::fprintf(stderr, "%s\n", sim.initError.c_str());
        std::exit(1);
    }
    g_log.clear();
    sim.steps(n);
    std::printf("%s: %s\n", name, g_log.c_str());
    if (sim.getSimTime().getTimestamp() != n) std::printf("%s: wrong time\n", name);
}

int main(int argc, char** argv) {
    const Options o = parse_options(argc, argv);
    drive<RealMovement, BasicInfection, DetailedTesting, NoClosure>("shipped", o, 26);
    drive<SelectableMovement, BasicInfection, SelectableTesting, SelectableClosure>("selectable", o, 26);
    drive<OwnMovement, BasicInfection, NoTesting, NoClosure>("movement", o, 2);
    drive<RealMovement, OwnInfection, NoTesting, NoClosure>("infection", o, 2);
    drive<RealMovement, MinimalInfection, NoTesting, NoClosure>("minimal", o, 2);
    drive<RealMovement, BasicInfection, NoTesting, OwnClosure>("closure", o, 2);
    drive<NamedMovement, BasicInfection, NoTesting, NoClosure>("named", o, 2);
    drive<RealMovement, BasicInfection, OwnTesting, NoClosure>("testing", o, 25);
}
