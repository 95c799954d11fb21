// Host side of the drop-in: the policy-templated Simulation<...> of the
// reference (include/simulation.h:53-976) with HIP-backed policies that call
// the C ABI of include/pansim_hip.h.  Same template parameters, same policy
// names and hook signatures (addProgramParameters / initializeArgs / init /
// planLocations / movement / infectionsAtLocations / performTests / midnight /
// step), same runSimulation and runForDay orderings.  Policies reach the
// device context through static_cast<SimulationType*>(this)->ctx, as the
// reference's policies reach agents/locs.
//
// Differences on purpose: options come as ps::Options (parsed with the same
// flag names and defaults as the reference's cxxopts registrations), the
// population lives in the device context instead of process-wide singletons
// (so several Simulation objects are independent replicas), and the weekday
// is (startDay + day) % 7 instead of wall-clock localtime arithmetic.
#pragma once
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdio>
#include <functional>
#include <iostream>
#include <memory>
#include <string>
#include <tuple>
#include <type_traits>
#include <vector>

#include "../../../include/pansim_hip.h"
#include "model.h"
#include "outputs.h"
#include "scenario.h"

namespace ps {

// Timehandler (include/tools/timeHandler.h:19-106): a step counter.
class Timehandler {
    unsigned counter_ = 0;
    unsigned timeStep_;
    unsigned stepsPerDay_;
    unsigned startDay_;
    unsigned startDate_;

public:
    Timehandler(unsigned timeStep, unsigned startDay, unsigned startDate)
        : timeStep_(timeStep), stepsPerDay_(1440u / timeStep), startDay_(startDay), startDate_(startDate) {}
    Timehandler& operator++() {
        ++counter_;
        return *this;
    }
    unsigned getTimestamp() const { return counter_; }
    unsigned getMinutes() const { return (counter_ % stepsPerDay_) * timeStep_; }
    unsigned getStepsPerDay() const { return stepsPerDay_; }
    unsigned getStepsUntilMidnight() const { return stepsPerDay_ - (counter_ % stepsPerDay_); }
    unsigned getTimeStep() const { return timeStep_; }
    unsigned getStartDate() const { return startDate_; }
    bool isMidnight() const { return counter_ % stepsPerDay_ == 0; }
    unsigned getDay() const { return (startDay_ + counter_ / stepsPerDay_) % 7; }  // 0 = Monday
};

inline void check(pansim_ctx* ctx, int rc, const char* what) {
    if (rc != 0) throw InitError(rc, std::string(what) + ": " + pansim_last_error(ctx));
}

// A policy class names itself in EngineHooks where calls of the engine that
// take several hooks together may stand for its own: a movement policy whose
// movement() is pansim_movement_step with stepParams(), an infection policy
// whose infectionsAtLocationsMask() is pansim_infection_step with
// dayInfectionParams() unless dumpsInfectiousList(), a closure policy whose
// step() does nothing (then Simulation::daySteps gives runs of steps to
// pansim_run_steps), a testing policy whose performTests() is
// pansim_testing_day with dayTests()' arguments and setStats() of its counts
// (then Simulation::dayUpdates gives a midnight to pansim_midnight_day).  A
// policy derived from one of these inherits the name of its base, not its own,
// so its hooks are called one by one, as any other policy's, unless it names
// itself too.
template <class P, class = void>
struct UsesEngineHooks : std::false_type {};
template <class P>
struct UsesEngineHooks<P, std::void_t<typename P::EngineHooks>> : std::is_same<typename P::EngineHooks, P> {};

// ---------------------------------------------------------------- movement
// NoMovement (include/policies/movementPolicies.h:9-20).  The midnight hook
// rebuilds the engine's per-location sums, which the midnight passes change
// (the reference recomputes them at every infection step).
template <typename SimulationType>
class NoMovement {
public:
    static void addProgramParameters(Options&) {}
    void initializeArgs(const Options&) {}
    void init(const LocationTypeIds&, unsigned) {}
    void planLocations(Timehandler, unsigned) {
        auto* self = static_cast<SimulationType*>(this);
        check(self->ctx, pansim_rebuild_locations(self->ctx), "planLocations");
    }
    void movement(Timehandler, unsigned) {}
};

// DummyMovement (include/policies/movementPolicies.h:22-65)
template <typename SimulationType>
class DummyMovement {
public:
    static void addProgramParameters(Options&) {}
    void initializeArgs(const Options&) {}
    void init(const LocationTypeIds&, unsigned) {}
    void planLocations(Timehandler, unsigned) {
        auto* self = static_cast<SimulationType*>(this);
        check(self->ctx, pansim_dummy_plan_locations(self->ctx), "planLocations");
    }
    void movement(Timehandler simTime, unsigned) {
        auto* self = static_cast<SimulationType*>(this);
        check(self->ctx, pansim_dummy_movement_step(self->ctx, simTime.getTimestamp()), "movement");
    }
};

// RealMovement (include/policies/movementPolicies.h:1339-1752)
template <typename SimulationType>
class RealMovement {
    unsigned quarantineLength = 10;

public:
    using EngineHooks = RealMovement;
    bool enableCurfew = false;
    unsigned curfewBegin = 0;
    unsigned curfewEnd = 0;
    bool curfewTimeConverted = false;
    unsigned schoolAgeRestriction = 99;
    bool holidayModeActive = false;
    bool quarantineImmuneActive = false;
    bool lockdownNonvaccActive = false;
    unsigned quarantinePolicy = 3;

    static void addProgramParameters(Options&) {}
    void initializeArgs(const Options& o) {
        quarantinePolicy = o.quarantinePolicy;
        quarantineLength = o.quarantineLength;
    }
    void init(const LocationTypeIds&, unsigned) {}

    pansim_step_params stepParams(const Timehandler& t, unsigned timeStep) const {
        pansim_step_params p{};
        p.timestamp = t.getTimestamp();
        p.time_step = timeStep;
        p.day_of_week = holidayModeActive ? 6u : t.getDay();
        p.quarantine_policy = quarantinePolicy;
        p.quarantine_length = quarantineLength;
        p.enable_curfew = enableCurfew ? 1u : 0u;
        p.curfew_begin = curfewBegin;
        p.curfew_end = curfewEnd;
        p.school_age_restriction = schoolAgeRestriction;
        p.quarantine_immune_active = quarantineImmuneActive ? 1u : 0u;
        p.lockdown_nonvacc_active = lockdownNonvaccActive ? 1u : 0u;
        return p;
    }

    // the arguments of the day's planning; curfew times set since are
    // converted to steps first
    pansim_step_params planParams(const Timehandler& simTime, unsigned timeStep) {
        if (!curfewTimeConverted) {
            curfewBegin = curfewBegin / timeStep;
            curfewEnd = curfewEnd / timeStep;
            curfewTimeConverted = true;
        }
        return stepParams(simTime, timeStep);
    }

    void planLocations(Timehandler simTime, unsigned timeStep) {
        auto* self = static_cast<SimulationType*>(this);
        pansim_step_params p = planParams(simTime, timeStep);
        check(self->ctx, pansim_plan_locations(self->ctx, &p), "planLocations");
    }

    void movement(Timehandler simTime, unsigned timeStep) {
        auto* self = static_cast<SimulationType*>(this);
        pansim_step_params p = stepParams(simTime, timeStep);
        check(self->ctx, pansim_movement_step(self->ctx, &p), "movement");
    }

    // movement and infection of n steps of one day as one engine call
    // (Simulation::daySteps, where nothing is looked at in between)
    bool stepsInRanges() const { return true; }
    void moveAndInfect(Timehandler simTime, unsigned timeStep, unsigned n, uint32_t mask, float k, float season) {
        auto* self = static_cast<SimulationType*>(this);
        pansim_step_params p = stepParams(simTime, timeStep);
        check(self->ctx, pansim_run_steps(self->ctx, &p, n, mask, k, season), "movement and infection");
    }
};

// ---------------------------------------------------------------- infection
// BasicInfection (include/policies/infectionPolicies.h:8-589)
template <typename SimulationType>
class BasicInfection {
    double k = 0.000347;
    double c0_offset = 3.08, trunc = 0.5;
    std::vector<int> d_offset;
    int d_peak_offset = 0;
    std::string dumpPath;  // --dumpLocationInfectiousList
    bool dumpEnabled = false;
    InfectiousListDump dump;

    // One infection pass of one variant with the dump on: the launch, then
    // the new infections and the infectious agents at their locations.
    void infectAndDump(const Timehandler& simTime, unsigned timeStep, uint32_t variant, float tmpK, float season) {
        auto* self = static_cast<SimulationType*>(this);
        pansim_ctx* ctx = self->ctx;
        if (!dumpEnabled) {
            check(ctx, pansim_infection_dump_enable(ctx, 1), "dumpLocationInfectiousList");
            dumpEnabled = true;
        }
        check(ctx, pansim_infection_step(ctx, simTime.getTimestamp(), 1u << variant, tmpK, season, timeStep),
              "infectionsAtLocations");
        size_t nNew = 0, nInf = 0;
        check(ctx, pansim_infection_dump_collect(ctx, nullptr, nullptr, 0, &nNew, nullptr, nullptr, nullptr, 0, &nInf),
              "dumpLocationInfectiousList");
        std::vector<uint32_t> na(nNew + 1), nl(nNew + 1), ia(nInf + 1), il(nInf + 1);
        std::vector<float> iv(nInf + 1);
        check(ctx, pansim_infection_dump_collect(ctx, na.data(), nl.data(), na.size(), &nNew, ia.data(), il.data(), iv.data(),
                                                 ia.size(), &nInf),
              "dumpLocationInfectiousList");
        na.resize(nNew);
        nl.resize(nNew);
        ia.resize(nInf);
        il.resize(nInf);
        iv.resize(nInf);
        dump.insert(simTime.getTimestamp(), variant, na, nl, ia, il, iv);
    }

public:
    using EngineHooks = BasicInfection;
    static void addProgramParameters(Options&) {}
    // infectionPolicies.h:110-114
    void finalize() {
        if (!dumpPath.empty()) dump.write(dumpPath);
    }

    void initializeArgs(const Options& o) {
        k = o.k;
        d_offset = split_int(o.d_offset, ',');
        d_peak_offset = o.d_peak_offset;
        c0_offset = o.c0;
        trunc = o.trunc;
        dumpPath = o.dumpLocationInfectiousList;
    }
    bool dumpsInfectiousList() const { return !dumpPath.empty(); }

    // infectionPolicies.h:443-478 (host, once per step)
    double seasonalityMultiplier(const Timehandler& simTime) const {
        unsigned simDay = simTime.getTimestamp() / simTime.getStepsPerDay();
        int d = (int)simTime.getStartDate() + (int)simDay;
        int d_peak = 59 + 22;
        d += 6;
        double c0 = 3.08;
        double trunc_val = 0.5;
        if (simDay > 250 && simDay < 450) {
            d += d_offset.empty() ? 0 : d_offset[0];
            d_peak += d_peak_offset;
            c0 = c0_offset;
        } else if (simDay > 600) {
            trunc_val = trunc;
            if (d_offset.size() > 1) d += d_offset[1];
        }
        int d_mod = d % 366;
        if (d_mod > 366 / 2) d_mod = 366 - d_mod;
        double normed = (0.5 * c0 * std::cos(2.0 * M_PI * (double)(d_mod - d_peak) / 366.0) + (1.0 - 0.5 * c0)) /
                        (0.5 * c0 * std::cos(2.0 * M_PI * (double)(d_peak - d_peak) / 366.0) + (1.0 - 0.5 * c0));
        double calc = std::min(std::max(normed, trunc_val), 1.0);
        if (d_mod < d_peak) return 1.0;
        return calc;
    }

    // All variants of `mask` in one pass (ascending variant order).
    void infectionsAtLocationsMask(const Timehandler& simTime, unsigned timeStep, uint32_t mask) {
        auto* self = static_cast<SimulationType*>(this);
        float tmpK = (float)k;
        float season = (float)seasonalityMultiplier(simTime);
        if (!dumpPath.empty()) {  // one pass per variant, each dumped (infectionPolicies.h:548-557)
            for (uint32_t v = 0; v < 32; ++v)
                if ((mask >> v) & 1u) infectAndDump(simTime, timeStep, v, tmpK, season);
            return;
        }
        check(self->ctx, pansim_infection_step(self->ctx, simTime.getTimestamp(), mask, tmpK, season, timeStep),
              "infectionsAtLocations");
    }
    void infectionsAtLocations(const Timehandler& simTime, unsigned timeStep, uint8_t variant) {
        infectionsAtLocationsMask(simTime, timeStep, 1u << variant);
    }
    // the arguments infectionsAtLocationsMask passes for this day (k and the
    // seasonality are constant within a day)
    void dayInfectionParams(const Timehandler& simTime, float& kOut, float& seasonOut) const {
        kOut = (float)k;
        seasonOut = (float)seasonalityMultiplier(simTime);
    }
};

// ---------------------------------------------------------------- testing
template <typename SimulationType>
class NoTesting {
public:
    using EngineHooks = NoTesting;
    static void addProgramParameters(Options&) {}
    void initializeArgs(const Options&) {}
    void init(const LocationTypeIds&) {}
    void performTests(Timehandler, unsigned) {}
    void dayTests(pansim_midnight& m) const { m.testing = 0; }
    void setStats(const uint32_t*) {}
    std::tuple<unsigned, unsigned, unsigned> getStats() { return {0u, 0u, 0u}; }
    void updateTestingProbs(const std::string&) {}
};

// DetailedTesting (include/policies/testingPolicies.h:292-476)
template <typename SimulationType>
class DetailedTesting {
    unsigned quarantineLength = 10;
    unsigned stats_[3] = {0, 0, 0};
    double probs_[6] = {0.005, 0.2, 0.1, 0.1, 0.2, 0.3};
    unsigned testingDelay = 5;
    bool usePCR = true;

public:
    using EngineHooks = DetailedTesting;
    static void addProgramParameters(Options&) {}
    void updateTestingProbs(const std::string& s) {
        auto p = split_double(s, ',');
        for (size_t i = 0; i < p.size() && i < 6; ++i) probs_[i] = p[i];
    }
    void initializeArgs(const Options& o) {
        testingDelay = o.testingRepeatDelay;
        updateTestingProbs(o.testingProbabilities);
        quarantineLength = o.quarantineLength;
        if (o.testingMethod == "PCR") usePCR = true;
        else if (o.testingMethod == "antigen") usePCR = false;
        else throw InitError(ERR_BAD_TESTING, "unrecognized testingMethod " + o.testingMethod + " must be either PCR or antigen");
    }
    void init(const LocationTypeIds&) {}
    std::tuple<unsigned, unsigned, unsigned> getStats() { return {stats_[0], stats_[1], stats_[2]}; }
    // performTests as part of a midnight's pass over the agents, and its counts
    void dayTests(pansim_midnight& m) const {
        m.testing = 1;
        for (int i = 0; i < 6; ++i) m.test_probs[i] = probs_[i];
        m.testing_delay = testingDelay;
        m.quarantine_length = quarantineLength;
        m.use_pcr = usePCR ? 1u : 0u;
    }
    void setStats(const uint32_t* t) {
        for (int i = 0; i < 3; ++i) stats_[i] = t[i];
    }
    void performTests(Timehandler simTime, unsigned timeStep) {
        auto* self = static_cast<SimulationType*>(this);
        uint32_t out[3];
        check(self->ctx,
              pansim_testing_day(self->ctx, simTime.getTimestamp(), timeStep, probs_, testingDelay, quarantineLength,
                                 usePCR ? 1u : 0u, out),
              "performTests");
        for (int i = 0; i < 3; ++i) stats_[i] = out[i];
    }
};

// ---------------------------------------------------------------- closures
template <typename SimulationType>
class NoClosure {
public:
    using EngineHooks = NoClosure;
    static void addProgramParameters(Options&) {}
    void initializeArgs(const Options&) {}
    void init(const LocationTypeIds&, const std::vector<ClosureRuleRaw>&, const std::string&) {}
    void midnight(Timehandler, unsigned, std::vector<unsigned>&) {}
    void step(Timehandler, unsigned) {}
};

// RuleClosure (include/policies/closurePolicies.h:47-481)
template <typename SimulationType>
class RuleClosure {
    struct GlobalCondition {
        std::vector<unsigned> headerPos;
        std::vector<double> history;
        int pos = 0;
        bool active = false;
        std::function<bool(GlobalCondition*, std::vector<unsigned>&)> condition;
    };
    struct Rule {
        std::string name;
        std::vector<size_t> conditions;
        std::function<void(Rule*)> rule;
        bool previousOpenState = true;
    };
    std::vector<GlobalCondition> globalConditions;
    std::vector<Rule> rules;
    unsigned enableClosures = 1;

    static std::vector<std::string> splitHeader(const std::string& h) {
        std::vector<std::string> out;
        std::string cur;
        for (char c : h) {
            if (c == '\t') {
                if (!cur.empty()) out.push_back(cur);
                cur.clear();
            } else cur.push_back(c);
        }
        if (!cur.empty()) out.push_back(cur);
        return out;
    }
    bool allActive(const Rule* r) const {
        bool close = true;
        for (size_t c : r->conditions) close = close && globalConditions[c].active;
        return close;
    }

public:
    using EngineHooks = RuleClosure;
    static void addProgramParameters(Options&) {}
    void initializeArgs(const Options& o) { enableClosures = o.enableClosures; }

    void init(const LocationTypeIds& lt, const std::vector<ClosureRuleRaw>& input, const std::string& statesHeader) {
        auto* self = static_cast<SimulationType*>(this);
        std::vector<std::string> header = splitHeader(statesHeader);
        std::vector<unsigned> hospitalStates;
        for (unsigned i = 0; i < header.size(); ++i)
            if (header[i].find("_h") != std::string::npos) hospitalStates.push_back(i);
        const unsigned numberOfAgents = self->sc.agents.n;
        static const char* always[] = {"Masks",          "Curfew",           "HolidayMode",      "SchoolAgeRestriction",
                                       "ExposeToMutation", "ReduceMovement", "QuarantinePolicy", "QuarantineImmune",
                                       "LockdownNonvacc",  "TestingProb"};
        globalConditions.reserve(input.size());
        rules.reserve(input.size());
        for (const auto& r : input) {
            bool keep = enableClosures != 0;
            for (auto* a : always) keep = keep || r.name == a;
            if (!keep) continue;
            GlobalCondition c;
            const int closeAfter = r.closeAfter, openAfter = r.openAfter;
            const double threshold = r.threshold, threshold2 = r.threshold2;
            // history window with hysteresis (closurePolicies.h:137-166)
            auto hysteresis = [threshold, threshold2, openAfter, closeAfter](GlobalCondition* g, double value) {
                g->history[g->pos] = value;
                const int hs = (int)g->history.size();
                g->pos = (g->pos + 1) % hs;
                auto wrap = [hs](int x) { return ((x % hs) + hs) % hs; };
                if (!g->active && value > threshold) {
                    bool below = false;
                    for (int i = wrap(g->pos - closeAfter); i != g->pos; i = (i + 1) % hs) below |= g->history[i] < threshold;
                    return below ? g->active : true;
                }
                if (g->active && value <= threshold2) {
                    bool above = false;
                    for (int i = wrap(g->pos - openAfter); i != g->pos; i = (i + 1) % hs) above |= g->history[i] >= threshold2;
                    return above ? g->active : false;
                }
                return g->active;
            };
            if (r.conditionType == "afterDays") {
                if (closeAfter >= 0 || openAfter <= 0)
                    throw InitError(ERR_BAD_CLOSURE, "For closure rule 'afterDays', closeAfter must be -1, openAfter must be >0");
                c.condition = [openAfter, threshold](GlobalCondition* g, std::vector<unsigned>&) {
                    int day = (int)g->history[0]++;
                    return day >= threshold && day < threshold + openAfter;
                };
                c.history.assign(1, 0.0);
            } else if (r.conditionType == "hospitalizedFraction") {
                if (closeAfter <= 0 || openAfter <= 0)
                    throw InitError(ERR_BAD_CLOSURE, "For closure rule 'hospitalizedFraction', closeAfter and openAfter must be >0");
                c.headerPos = hospitalStates;
                c.condition = [hysteresis, numberOfAgents](GlobalCondition* g, std::vector<unsigned>& s) {
                    double accum = 0.0;
                    for (unsigned p : g->headerPos) accum += s[p];
                    return hysteresis(g, accum / (double)numberOfAgents);
                };
                c.history.assign(std::max(closeAfter, openAfter) + 2, 0.0);
            } else if (r.conditionType == "newDeadFraction") {
                if (closeAfter <= 0 || openAfter <= 0)
                    throw InitError(ERR_BAD_CLOSURE, "For closure rule 'newDeadFraction', closeAfter and openAfter must be >0");
                for (unsigned i = 0; i < header.size(); i++)
                    if (header[i] == "D1") c.headerPos.push_back(i);
                c.headerPos.push_back(0);
                c.condition = [hysteresis, numberOfAgents](GlobalCondition* g, std::vector<unsigned>& s) {
                    double value = (s[g->headerPos[0]] - g->headerPos[1]) / (double)numberOfAgents;
                    g->headerPos[1] = s[g->headerPos[0]];
                    return hysteresis(g, value);
                };
                c.history.assign(std::max(closeAfter, openAfter) + 2, 0.0);
            } else {
                throw InitError(ERR_BAD_CLOSURE, "Unknown closure type " + r.conditionType);
            }
            globalConditions.push_back(c);
            Rule rule;
            rule.name = r.name;
            rule.conditions = {globalConditions.size() - 1};
            if (r.name == "Masks") {
                double coef = std::atof(r.parameter.c_str());
                rule.rule = [this, self, coef](Rule* rr) {
                    bool open = !allActive(rr);
                    if (rr->previousOpenState != open) {
                        self->currentMaskValue = open ? 1.0 : coef;
                        check(self->ctx, pansim_scale_infectiousness(self->ctx, coef, open ? 1u : 0u), "Masks");
                        rr->previousOpenState = open;
                    }
                };
            } else if (r.name == "Curfew") {
                unsigned cb = 0, ce = 0;
                if (r.parameter.size() == 9) {
                    cb = (unsigned)std::atoi(r.parameter.substr(0, 2).c_str()) * 60 + (unsigned)std::atoi(r.parameter.substr(2, 2).c_str());
                    ce = (unsigned)std::atoi(r.parameter.substr(5, 2).c_str()) * 60 + (unsigned)std::atoi(r.parameter.substr(7, 2).c_str());
                } else if (!r.parameter.empty())
                    throw InitError(ERR_BAD_CLOSURE, "curfew parameter string needs to be exactly 9 characters long");
                rule.rule = [this, self, cb, ce](Rule* rr) {
                    bool close = allActive(rr);
                    if (rr->previousOpenState != !close) {
                        self->toggleCurfew(close, cb, ce);
                        rr->previousOpenState = !close;
                    }
                };
            } else if (r.name == "HolidayMode" || r.name == "QuarantineImmune" || r.name == "LockdownNonvacc") {
                int which = r.name == "HolidayMode" ? 0 : (r.name == "QuarantineImmune" ? 1 : 2);
                rule.rule = [this, self, which](Rule* rr) {
                    bool close = allActive(rr);
                    if (rr->previousOpenState != !close) {
                        if (which == 0) self->toggleHolidayMode(close);
                        else if (which == 1) self->toggleQuarantineImmune(close);
                        else self->toggleLockdownNonvacc(close);
                        rr->previousOpenState = !close;
                    }
                };
            } else if (r.name == "QuarantinePolicy") {
                int qp = std::atoi(r.parameter.c_str());
                rule.rule = [this, self, qp](Rule* rr) {
                    bool close = allActive(rr);
                    if (close) {
                        self->quarantinePolicy((unsigned)qp);
                        rr->previousOpenState = close;
                    }
                };
            } else if (r.name == "SchoolAgeRestriction") {
                unsigned limit = (unsigned)std::atoi(r.parameter.c_str());
                rule.rule = [this, self, limit](Rule* rr) {
                    bool close = allActive(rr);
                    if (rr->previousOpenState != !close) {
                        self->setSchoolAgeRestriction(close ? limit : 99);
                        rr->previousOpenState = !close;
                    }
                };
            } else if (r.name == "ExposeToMutation") {
                double fraction = std::atof(r.parameter.c_str());
                unsigned variantIdx = (unsigned)(int)threshold2;
                if (variantIdx >= self->sc.variantMultiplier.size())
                    throw InitError(ERR_BAD_CLOSURE,
                                    "More ExposeToMutation events defined than infectiousnessMultiplier specified on the command line");
                rule.rule = [this, self, fraction, variantIdx](Rule* rr) {
                    if (!allActive(rr)) return;
                    check(self->ctx,
                          pansim_expose_mutation(self->ctx, self->getSimTime().getTimestamp(), variantIdx, fraction),
                          "ExposeToMutation");
                };
            } else if (r.name == "ReduceMovement") {
                double fraction = std::atof(r.parameter.c_str());
                unsigned homeType = lt.home;
                rule.rule = [this, self, fraction, homeType](Rule* rr) {
                    bool open = !allActive(rr);
                    if (rr->previousOpenState != open) {
                        self->reduceMovement(fraction, homeType, !open);
                        rr->previousOpenState = open;
                    }
                };
            } else if (r.name == "TestingProb") {
                std::string probs = r.parameter;
                rule.rule = [this, self, probs](Rule* rr) {
                    if (allActive(rr)) self->updateTestingProbs(probs);
                };
            } else {
                std::vector<uint32_t> toClose;
                for (int tt : r.locationTypesToClose) toClose.push_back((uint32_t)tt);
                if (toClose.size() >= 10)
                    throw InitError(ERR_BAD_CLOSURE, "Error, Closure Rule " + r.name + " has over 10 location types to close");
                rule.rule = [this, self, toClose](Rule* rr) {
                    bool open = !allActive(rr);
                    if (rr->previousOpenState != open) {
                        check(self->ctx, pansim_set_open_by_type(self->ctx, toClose.data(), (uint32_t)toClose.size(), open ? 1u : 0u),
                              "closure rule");
                        rr->previousOpenState = open;
                    }
                };
            }
            rules.push_back(rule);
        }
    }

    void midnight(Timehandler, unsigned, std::vector<unsigned>& stats) {
        for (auto& c : globalConditions) c.active = c.condition(&c, stats);
        for (auto& r : rules) r.rule(&r);
    }
    void step(Timehandler, unsigned) {}
};

// ---------------------------------------------------------------- state types
// Marker types for the PPState / AgentMeta template parameters: the state
// record (dynamicPPState.h) and agent metadata (agentMeta.h) live in device
// SoA arrays; these expose their static API.
struct DynamicPPState {
    static unsigned getNumberOfStates(const Scenario& sc) { return (unsigned)sc.st.names.size(); }
    static std::vector<std::string> getStateNames(const Scenario& sc) { return sc.st.names; }
};
struct BasicAgentMeta {};

// ---------------------------------------------------------------- simulation
template <typename PositionType, typename TypeOfLocation, typename PPState, typename AgentMeta,
          template <typename> class MovementPolicy, template <typename> class InfectionPolicy,
          template <typename> class TestingPolicy, template <typename> class ClosurePolicy>
class Simulation
    : public MovementPolicy<Simulation<PositionType, TypeOfLocation, PPState, AgentMeta, MovementPolicy, InfectionPolicy,
                                       TestingPolicy, ClosurePolicy>>,
      public InfectionPolicy<Simulation<PositionType, TypeOfLocation, PPState, AgentMeta, MovementPolicy, InfectionPolicy,
                                        TestingPolicy, ClosurePolicy>>,
      public TestingPolicy<Simulation<PositionType, TypeOfLocation, PPState, AgentMeta, MovementPolicy, InfectionPolicy,
                                      TestingPolicy, ClosurePolicy>>,
      public ClosurePolicy<Simulation<PositionType, TypeOfLocation, PPState, AgentMeta, MovementPolicy, InfectionPolicy,
                                      TestingPolicy, ClosurePolicy>> {
public:
    using Self = Simulation;
    using Movement = MovementPolicy<Self>;
    using Infection = InfectionPolicy<Self>;
    using Testing = TestingPolicy<Self>;
    using Closure = ClosurePolicy<Self>;

    Scenario sc;
    ModelArrays model;
    pansim_ctx* ctx = nullptr;
    unsigned timeStep;
    unsigned lengthOfSimulationWeeks;
    bool succesfullyInitialized = true;
    std::string statesHeader;
    int enableOtherDisease = 1;
    double currentMaskValue = 1.0;
    unsigned homeType = 2;
    unsigned immunizedToday = 0;
    bool print = true;
    std::vector<std::vector<unsigned>> dayStats;  // every statistics vector computed at a midnight
    std::vector<unsigned> variantCounts;
    std::string initError;
    int initErrorCode = 0;

    explicit Simulation(const Options& o, bool printOutput = true, uint32_t replica = 0)
        : timeStep(o.deltat), lengthOfSimulationWeeks(o.weeks), print(printOutput), simTime_(o.deltat ? o.deltat : 10, o.startDay, o.startDate) {
        try {
            sc = build_scenario(o);
            enableOtherDisease = o.otherDisease;
            Infection::initializeArgs(o);
            Movement::initializeArgs(o);
            Testing::initializeArgs(o);
            Closure::initializeArgs(o);
            build_model(sc, model);
            int rc = pansim_create(&ctx, &model.dims, &model.tables, &model.locations, &model.agents, o.seed, replica,
                                   timeStep, o.quarantinePolicy, o.quarantineLength);
            if (rc != 0) throw InitError(rc, std::string("pansim_create: ") + pansim_create_error());
            {  // Immunization::initCategories (immunization.h:229-420)
                int32_t order[10];
                for (int g = 0; g < 10; ++g) order[g] = sc.vacc.order[g];
                check(ctx, pansim_vaccination_init(ctx, order, sc.vacc.groupLevel.data()), "initCategories");
            }
            Movement::init(sc.lt, sc.locs.cemetery);
            Testing::init(sc.lt);
            statesHeader = sc.statesHeader;
            homeType = sc.lt.home;
            Closure::init(sc.lt, sc.rules, statesHeader);
            variantCounts.assign(sc.variantMultiplier.size(), 0);
            schedulesHost_ = sc.sched.events;
            offsetsHost_ = sc.sched.eventOffset;
            if (print) std::cout << statesHeader << '\n';
        } catch (const InitError& e) {
            succesfullyInitialized = false;
            initError = e.what();
            initErrorCode = e.code;
            if (print) std::cerr << e.what() << '\n';
        } catch (const std::exception& e) {
            succesfullyInitialized = false;
            initError = e.what();
            initErrorCode = ERR_BAD_DATA;
            if (print) std::cerr << e.what() << '\n';
        }
    }
    ~Simulation() {
        if (ctx) pansim_destroy(ctx);
    }
    Simulation(const Simulation&) = delete;
    Simulation& operator=(const Simulation&) = delete;

    Timehandler& getSimTime() { return simTime_; }

    // simulation.h:425-471
    void updateAgents(Timehandler& t) { check(ctx, pansim_progression_day(ctx, t.getTimestamp(), timeStep), "updateAgents"); }

    // the susceptibility pass's parameters (options: parsed once)
    void immunizationParams(pansim_midnight& m) {
        if (!immReady_) {
            const std::string* lists[6] = {&sc.opt.protectionInfection,       &sc.opt.protectionInfectionWaning,
                                           &sc.opt.protectionSymptomatic,     &sc.opt.protectionSymptomaticWaning,
                                           &sc.opt.protectionHospitalization, &sc.opt.protectionHospitalizationWaning};
            for (int l = 0; l < 6; ++l) {
                const auto v = split_float(*lists[l], ',');
                if (v.size() < 10) throw InitError(ERR_BAD_ARG, "protection parameters need 10 values");
                for (int i = 0; i < 10; ++i) imm_.protection[10 * l + i] = v[i];
            }
            auto vs = split_int(sc.opt.variantSimilarity, ',');
            auto vm = split_float(sc.opt.variantSimilarMultiplier, ',');
            for (size_t i = 0; i < vs.size() && i < 7; ++i) imm_.similarity[i] = vs[i];
            for (size_t i = 0; i < vm.size() && i < 7; ++i) imm_.similar_multiplier[i] = vm[i];
            immReady_ = true;
        }
        for (int i = 0; i < 60; ++i) m.protection[i] = imm_.protection[i];
        for (int i = 0; i < 7; ++i) {
            m.similarity[i] = imm_.similarity[i];
            m.similar_multiplier[i] = imm_.similar_multiplier[i];
        }
    }

    // Immunization::update (immunization.h:481-900): the susceptibility pass,
    // the booster rounds, then the first doses.
    void immunizationUpdate(Timehandler& t) {
        pansim_midnight m{};
        immunizationParams(m);
        check(ctx, pansim_immunization_day(ctx, t.getTimestamp(), timeStep, m.protection, m.similarity, m.similar_multiplier),
              "immunization");
        vaccinationRollout(t);
    }

    // initAgeGroups (immunization.h:421-479): booster shares per age group
    void initAgeGroups() {
        ageGroupsReady_ = true;
        uint32_t ages[10];
        check(ctx, pansim_age_group_counts(ctx, ages), "initAgeGroups");
        const auto& v = sc.vacc;
        ageGroupFrac_.assign(v.boosterStart.size(), std::array<float, 10>{});
        for (size_t r = 0; r < v.boosterStart.size(); ++r) {
            unsigned size[10], sum = 0;
            for (int g = 0; g < 10; ++g) {
                size[g] = (unsigned)((float)ages[g] * v.boosterAgePercent[r][g]);
                sum += size[g];
            }
            for (int g = 0; g < 10; ++g) ageGroupFrac_[r][g] = (float)size[g] / (float)sum;
        }
    }

    // numberOfBoostersToday / numberOfVaccinesToday (immunization.h:62-89)
    unsigned boostersToday(unsigned day, size_t r) const {
        const auto& v = sc.vacc;
        if ((int)day < v.boosterStart[r]) return 0;
        if (v.boosterPerWeek[r].empty()) return v.dailyBoosters;
        unsigned week = (day - (unsigned)v.boosterStart[r]) / 7;
        const auto& w = v.boosterPerWeek[r];
        return (unsigned)(w[week >= w.size() ? w.size() - 1 : week] / 7.0);
    }
    unsigned dosesToday(unsigned day) const {
        const auto& v = sc.vacc;
        if (day < v.startDay) return 0;
        if (v.vaccPerWeek.empty()) return v.dailyDoses;
        unsigned week = (day - v.startDay) / 7;
        return (unsigned)(v.vaccPerWeek[week >= v.vaccPerWeek.size() ? v.vaccPerWeek.size() - 1 : week] / 7.0);
    }
    // whether the rollout of the day gives (or may give) any dose
    bool rolloutToday(const Timehandler& t) const {
        const unsigned day = t.getTimestamp() / t.getStepsPerDay();
        for (size_t r = 0; r < sc.vacc.boosterStart.size(); ++r)
            if (boostersToday(day, r) > 0) return true;
        return currentCategory_ < 10 && dosesToday(day) > 0;
    }

    // the rollout
    void vaccinationRollout(Timehandler& t) {
        if (!ageGroupsReady_) initAgeGroups();
        const unsigned ts = t.getTimestamp();
        const unsigned day = ts / t.getStepsPerDay();
        for (size_t r = 0; r < sc.vacc.boosterStart.size(); ++r)
            check(ctx, pansim_booster_round(ctx, ts, timeStep, (uint32_t)r, boostersToday(day, r), ageGroupFrac_[r].data()),
                  "boosters");
        uint32_t today = 0;
        check(ctx, pansim_vaccinate(ctx, ts, timeStep, dosesToday(day), &currentCategory_, &today), "vaccination");
        immunizedToday = today;
    }

    // simulation.h:169-204, host part: the factor of the day's admission
    // probabilities, 0 without a hospitalisation target
    bool hospitalTarget(const Timehandler& t) const {
        return t.getTimestamp() / t.getStepsPerDay() < sc.totalHospitalizations.size();
    }
    float otherDiseaseFactor(Timehandler& t) {
        if (!hospitalTarget(t)) return 0.0f;
        unsigned simDay = t.getTimestamp() / t.getStepsPerDay();
        uint32_t inHosp = 0;
        check(ctx, pansim_count_hospitalized_covid(ctx, t.getTimestamp(), sc.opt.dueWithCOVID, &inHosp), "otherDisease");
        unsigned target = (unsigned)std::max(0.0, double(sc.totalHospitalizations[simDay]) - double(inHosp) * (9730000.0 / 179500.0));
        return float(target) / 48000.0;
    }
    void otherDisease(Timehandler& t) {
        check(ctx, pansim_other_disease_day(ctx, t.getTimestamp(), timeStep, otherDiseaseFactor(t)), "otherDisease");
    }

    // The routines of a midnight up to the statistics (testing, progression,
    // immunity, other disease, statistics) as one pass over the agents.
    // fillMidnight: its arguments; false where something goes between them.
    bool fillMidnight(const Timehandler& t, pansim_midnight& m) {
        if constexpr (UsesEngineHooks<Testing>::value) {
            if (rolloutToday(t) || (enableOtherDisease && hospitalTarget(t))) return false;
            firstMidnightHalf(t, m);
            secondMidnightHalf(t, m, 0.0f);
            m.count_immunized = 1;
            return true;
        }
        return false;
    }
    void firstMidnightHalf(const Timehandler& t, pansim_midnight& m) {
        m.timestamp = t.getTimestamp();
        m.time_step = timeStep;
        if constexpr (UsesEngineHooks<Testing>::value)
            if (t.getTimestamp() > 0) Testing::dayTests(m);
        m.progression = t.getTimestamp() > 0 ? 1u : 0u;
        m.immunization = 1;
        immunizationParams(m);
    }
    void secondMidnightHalf(const Timehandler& t, pansim_midnight& m, float probabilityMul) {
        m.timestamp = t.getTimestamp();
        m.time_step = timeStep;
        m.other_disease = enableOtherDisease ? 1u : 0u;
        m.probability_mul = probabilityMul;
        m.statistics = 1;
        if (!m.testing) {
            auto ts = Testing::getStats();
            m.tests[0] = std::get<0>(ts), m.tests[1] = std::get<1>(ts), m.tests[2] = std::get<2>(ts);
        }
        m.immunized = immunizedToday;
    }
    std::vector<unsigned> takeMidnight(const pansim_midnight& m, bool printLine = true) {
        if constexpr (UsesEngineHooks<Testing>::value)
            if (m.testing) Testing::setStats(m.tests);
        immunizedToday = m.immunized;
        std::vector<unsigned> stats(m.stats, m.stats + m.stats_len);
        if (printLine && print) printStats(stats);
        return stats;
    }
    std::vector<unsigned> dayUpdates(Timehandler& t) {
        if constexpr (UsesEngineHooks<Testing>::value) {
            pansim_midnight m{};
            if (!fillMidnight(t, m)) {
                firstMidnightHalf(t, m);
                check(ctx, pansim_midnight_day(ctx, &m), "midnight");
                if (m.testing) Testing::setStats(m.tests);
                vaccinationRollout(t);
                const float mul = enableOtherDisease ? otherDiseaseFactor(t) : 0.0f;
                m = pansim_midnight{};
                secondMidnightHalf(t, m, mul);
            }
            check(ctx, pansim_midnight_day(ctx, &m), "midnight");
            return takeMidnight(m);
        } else {
            if (t.getTimestamp() > 0) Testing::performTests(t, timeStep);
            if (t.getTimestamp() > 0) updateAgents(t);
            immunizationUpdate(t);
            if (enableOtherDisease) otherDisease(t);
            return refreshAndPrintStatistics(t);
        }
    }

    std::vector<unsigned> refreshAndPrintStatistics(Timehandler& t, bool printLine = true) {
        auto ts = Testing::getStats();
        uint32_t test[3] = {std::get<0>(ts), std::get<1>(ts), std::get<2>(ts)};
        std::vector<uint32_t> out(512);
        size_t len = 0;
        check(ctx, pansim_stats_day(ctx, t.getTimestamp(), timeStep, test, immunizedToday, out.data(), out.size(), &len), "statistics");
        out.resize(len);
        std::vector<unsigned> stats(out.begin(), out.end());
        if (printLine && print) printStats(stats);
        return stats;
    }

    std::vector<unsigned> countVariantCases() {
        std::vector<uint32_t> out(7, 0);
        check(ctx, pansim_count_variants(ctx, out.data()), "countVariantCases");
        return std::vector<unsigned>(out.begin(), out.begin() + sc.variantMultiplier.size());
    }

    uint32_t activeMask() const {
        uint32_t m = 0;
        for (size_t v = 0; v < variantCounts.size(); ++v)
            if (variantCounts[v] > 0) m |= 1u << v;
        return m;
    }

    void midnight() {
        Timehandler& t = simTime_;
        closeDay(dayUpdates(t));
        Movement::planLocations(t, timeStep);
        variantCounts = countVariantCases();
    }
    // a midnight's statistics: recorded, then the closure rules act on them
    void closeDay(std::vector<unsigned> stats) {
        dayStats.push_back(stats);
        Closure::midnight(simTime_, timeStep, stats);
    }

    // The parts of one step that a replica batch (pansim_amd/csrc/host/ensemble.h)
    // runs per replica around its batched movement and infection launches.
    pansim_step_params batchPlanParams() { return Movement::planParams(simTime_, timeStep); }
    pansim_step_params batchStepParams() const { return Movement::stepParams(simTime_, timeStep); }
    void batchInfectionParams(uint32_t& mask, float& kOut, float& seasonOut) const {
        mask = activeMask();
        Infection::dayInfectionParams(simTime_, kOut, seasonOut);
    }
    void finishBatchedStep() {
        Closure::step(simTime_, timeStep);
        ++simTime_;
    }

    // One and n iterations of runSimulation's loop (simulation.h:904-923).
    void step() { steps(1); }
    void steps(unsigned n) {
        while (n > 0) {
            if (simTime_.isMidnight()) midnight();
            const unsigned spd = simTime_.getStepsPerDay();
            const unsigned m = std::min(n, spd - simTime_.getTimestamp() % spd);
            daySteps(m);
            n -= m;
        }
    }

    // n steps of the present day, after its midnight block: hook by hook, or
    // as one engine call where none of the hooks does anything that it does
    // not (k and the seasonality are the day's).
    void daySteps(unsigned n) {
        if constexpr (UsesEngineHooks<Movement>::value && UsesEngineHooks<Infection>::value && UsesEngineHooks<Closure>::value) {
            if (Movement::stepsInRanges() && !Infection::dumpsInfectiousList()) {
                float k, season;
                Infection::dayInfectionParams(simTime_, k, season);
                Movement::moveAndInfect(simTime_, timeStep, n, activeMask(), k, season);
                for (unsigned i = 0; i < n; ++i) ++simTime_;
                return;
            }
        }
        for (unsigned i = 0; i < n; ++i) {
            Movement::movement(simTime_, timeStep);
            Closure::step(simTime_, timeStep);
            Infection::infectionsAtLocationsMask(simTime_, timeStep, activeMask());
            ++simTime_;
        }
    }

    // simulation.h:899-926
    void runSimulation() {
        if (!succesfullyInitialized) return;
        const unsigned total = lengthOfSimulationWeeks * 7u * simTime_.getStepsPerDay();
        if (simTime_.getTimestamp() < total) steps(total - simTime_.getTimestamp());
        printAgentStatJSON();
        Infection::finalize();
    }

    // simulation.h:958-961 (the day interface's end)
    void finalize() {
        if (!succesfullyInitialized) return;
        printAgentStatJSON();
        Infection::finalize();
    }

    // AgentList::printAgentStatJSON (agentsList.h:280-327): the --outAgentStat
    // JSON, then with --diags > 0 the summary on stdout.
    void printAgentStatJSON() {
        if (sc.opt.outAgentStat.empty() && sc.opt.diags == 0) return;
        AgentStatColumns c;
        const uint32_t ts = simTime_.getTimestamp();
        auto get = [&](const char* name, std::vector<uint32_t>& v) {
            v.resize(sc.agents.n);
            check(ctx, pansim_download_field(ctx, name, ts, v.data(), v.size()), "printAgentStatJSON");
        };
        get("infectedTimestamp", c.infectedTimestamp);
        get("infectedCount", c.infectedCount);
        get("statsVariant", c.variant);
        get("infectedLocation", c.infectedLocation);
        get("diagnosedTimestamp", c.diagnosedTimestamp);
        get("quarantinedTimestamp", c.quarantinedTimestamp);
        get("quarantinedUntilTimestamp", c.quarantinedUntilTimestamp);
        get("daysInQuarantine", c.daysInQuarantine);
        get("hospitalizedTimestamp", c.hospitalizedTimestamp);
        get("hospitalizedUntilTimestamp", c.hospitalizedUntilTimestamp);
        get("immunizationTimestamp", c.immunizationTimestamp);
        get("immunizationCount", c.immunizationCount);
        get("recoveredTimestamp", c.recoveredTimestamp);
        get("worstState", c.worstState);
        get("worstStateTimestamp", c.worstStateTimestamp);
        get("worstStateEndTimestamp", c.worstStateEndTimestamp);
        write_agent_stats_json(sc.opt.outAgentStat, c, sc.st.names);
        if (sc.opt.diags > 0)
            print_agent_stat_diags(std::cout, c, sc.agents.age, sc.locs.type, sc.locs.cemetery, sc.lt.types.size() + 1);
    }

    // simulation.h:928-956
    std::vector<unsigned> runForDay(const std::vector<std::string>& flags) {
        processFlags(flags);
        auto stats = refreshAndPrintStatistics(simTime_, false);
        Closure::midnight(simTime_, timeStep, stats);
        Movement::planLocations(simTime_, timeStep);
        variantCounts = countVariantCases();
        // (each day's steps apart: runForDay may start mid-day.  The dummy and
        // no-movement policies then run on over the midnight; RealMovement,
        // whose day needs a planning, reports its absence there.)
        for (unsigned left = simTime_.getStepsPerDay(); left > 0;) {
            const unsigned spd = simTime_.getStepsPerDay();
            const unsigned m = std::min(left, spd - simTime_.getTimestamp() % spd);
            daySteps(m);
            left -= m;
        }
        stats = dayUpdates(simTime_);
        dayStats.push_back(stats);
        check(ctx, pansim_rebuild_locations(ctx), "runForDay");
        return stats;
    }

    // simulation.h:779-897
    void processFlags(const std::vector<std::string>& flags) {
        for (const auto& flag : flags) {
            std::string prefix = flag.substr(0, 2);
            if (prefix == "TP") {
                if (flag == "TPdef") updateTestingProbs("0.00005,0.01,0.0005,0.0005,0.005,0.05");
                else if (flag == "TP015") updateTestingProbs("0.00005,0.2,0.04,0.04,0.005,0.05");
                else if (flag == "TP035") updateTestingProbs("0.00005,1.0,0.2,0.2,0.005,0.05");
            } else if (prefix == "PL") {
                const uint32_t fix[4] = {5, 6, 22, 44};
                if (flag == "PLNONE") check(ctx, pansim_set_open_by_type(ctx, fix, 4, 1), "PLNONE");
                else if (flag == "PL0") check(ctx, pansim_set_open_by_type(ctx, fix, 4, 0), "PL0");
            } else if (prefix == "CF") {
                if (flag == "CFNONE") toggleCurfew(false, 0, 0);
                else if (flag == "CF2000-0500") toggleCurfew(true, 20 * 60, 5 * 60);
            } else if (prefix == "SO") {
                if (flag == "SONONE") setSchoolAgeRestriction(99);
                else if (flag == "SO12") setSchoolAgeRestriction(12);
                else if (flag == "SO3") setSchoolAgeRestriction(3);
            } else if (prefix == "QU") {
                if (flag == "QU0") quarantinePolicy(0);
                else if (flag == "QU1") quarantinePolicy(1);
                else if (flag == "QU2") quarantinePolicy(2);
                else if (flag == "QU3") quarantinePolicy(3);
            } else if (prefix == "MA") {
                if (flag == "MA1.0" && currentMaskValue != 1.0) {
                    check(ctx, pansim_scale_infectiousness(ctx, currentMaskValue, 1), "MA1.0");
                    currentMaskValue = 1.0;
                } else if (flag == "MA0.8" && currentMaskValue != 0.8) {
                    currentMaskValue = 0.8;
                    check(ctx, pansim_scale_infectiousness(ctx, 0.8, 0), "MA0.8");
                }
            }
        }
    }

    void toggleCurfew(bool enable, unsigned begin, unsigned end) {
        Movement::enableCurfew = enable;
        Movement::curfewBegin = begin;
        Movement::curfewEnd = end;
        Movement::curfewTimeConverted = false;
    }
    void setSchoolAgeRestriction(unsigned limit) { Movement::schoolAgeRestriction = limit; }
    void toggleHolidayMode(bool enable) { Movement::holidayModeActive = enable; }
    void toggleQuarantineImmune(bool enable) { Movement::quarantineImmuneActive = enable; }
    void toggleLockdownNonvacc(bool enable) { Movement::lockdownNonvaccActive = enable; }
    void quarantinePolicy(unsigned qp) { Movement::quarantinePolicy = qp; }
    void updateTestingProbs(const std::string& probs) { Testing::updateTestingProbs(probs); }

    // AgentTypeList::setStayHome / unsetStayHome (src/agentData/agentType.cpp:42-109)
    void reduceMovement(double probability, unsigned homeT, bool set) {
        auto& off = offsetsHost_;
        auto& ev = schedulesHost_;
        auto same = [](const Event& a, const Event& b) { return a.start_h == b.start_h && a.start_m == b.start_m; };
        for (unsigned s = 0; s + 1 < off.size(); s++) {
            unsigned ws = off[s], we = ws;
            while (ws < off[s + 1]) {
                while (we < ev.size() && same(ev[we], ev[ws])) we++;
                if (!set) {
                    for (unsigned i = ws; i < we; i++)
                        if (ev[i].locType != homeT) ev[i].chance = (float)(ev[i].chance / (1.0 - probability));
                    for (unsigned i = ws; i < we; i++)
                        if (ev[i].locType == homeT) {
                            ev[i].chance = (float)((ev[i].chance - probability) / (1.0 - probability));
                            if (std::abs(ev[i].chance) < 1e-10) {
                                ev.erase(ev.begin() + i);
                                for (size_t j = s + 1; j < off.size(); j++) off[j]--;
                            }
                            break;
                        }
                } else {
                    bool home = false;
                    for (unsigned i = ws; i < we; i++)
                        if (ev[i].locType == homeT) {
                            home = true;
                            ev[i].chance = (float)(ev[i].chance + (1.0 - ev[i].chance) * probability);
                            break;
                        }
                    if (home && we - ws == 1) {
                        ws = we;
                        continue;
                    }
                    if (!home) {
                        Event h = ev[ws];
                        h.locType = homeT;
                        h.chance = (float)probability;
                        ev.insert(ev.begin() + ws, h);
                        we++;
                        for (size_t j = s + 1; j < off.size(); j++) off[j]++;
                    }
                    for (unsigned i = ws; i < we; i++)
                        if (ev[i].locType != homeT) ev[i].chance = (float)(ev[i].chance * (1.0 - probability));
                }
                ws = we;
            }
        }
        auto cev = to_c_events(ev);
        check(ctx, pansim_upload_schedules(ctx, off.data(), (uint32_t)off.size(), cev.data(), (uint32_t)cev.size()),
              "ReduceMovement");
    }

    void printStats(const std::vector<unsigned>& s) const {
        for (size_t i = 0; i < s.size(); ++i) std::cout << s[i] << (i + 1 < s.size() ? "\t" : "\n");
    }

private:
    Timehandler simTime_;
    uint32_t currentCategory_ = 0;
    bool ageGroupsReady_ = false;
    pansim_midnight imm_{};  // immunizationParams
    bool immReady_ = false;
    std::vector<std::array<float, 10>> ageGroupFrac_;
    std::vector<Event> schedulesHost_;
    std::vector<uint32_t> offsetsHost_;
};

// RealMovement with the movement policy chosen at run time (--movementPolicy):
// one library serves the three bindings the reference compiles separately.
// The knobs the closure rules set stay those of RealMovement.
template <typename SimulationType>
class SelectableMovement : public RealMovement<SimulationType> {
    using Real = RealMovement<SimulationType>;
    enum Mode { REAL, DUMMY, NONE } mode_ = REAL;

public:
    using EngineHooks = SelectableMovement;
    void initializeArgs(const Options& o) {
        Real::initializeArgs(o);
        mode_ = o.movementPolicy == "dummy" ? DUMMY : o.movementPolicy == "none" ? NONE : REAL;
    }
    bool realMovement() const { return mode_ == REAL; }
    bool stepsInRanges() const { return mode_ == REAL; }
    void planLocations(Timehandler simTime, unsigned timeStep) {
        auto* self = static_cast<SimulationType*>(this);
        if (mode_ == REAL) Real::planLocations(simTime, timeStep);
        else if (mode_ == DUMMY) check(self->ctx, pansim_dummy_plan_locations(self->ctx), "planLocations");
        else check(self->ctx, pansim_rebuild_locations(self->ctx), "planLocations");
    }
    void movement(Timehandler simTime, unsigned timeStep) {
        auto* self = static_cast<SimulationType*>(this);
        if (mode_ == REAL) Real::movement(simTime, timeStep);
        else if (mode_ == DUMMY) check(self->ctx, pansim_dummy_movement_step(self->ctx, simTime.getTimestamp()), "movement");
    }
};

// DetailedTesting or NoTesting, chosen at run time (--testingPolicy).
template <typename SimulationType>
class SelectableTesting : public DetailedTesting<SimulationType> {
    using Detailed = DetailedTesting<SimulationType>;
    NoTesting<SimulationType> none_;
    bool detailed_ = true;

public:
    using EngineHooks = SelectableTesting;
    void initializeArgs(const Options& o) {
        detailed_ = o.testingPolicy != "none";
        if (detailed_) Detailed::initializeArgs(o);
        else none_.initializeArgs(o);
    }
    void init(const LocationTypeIds& lt) {
        if (detailed_) Detailed::init(lt);
        else none_.init(lt);
    }
    void performTests(Timehandler simTime, unsigned timeStep) {
        if (detailed_) Detailed::performTests(simTime, timeStep);
        else none_.performTests(simTime, timeStep);
    }
    void dayTests(pansim_midnight& m) const {
        if (detailed_) Detailed::dayTests(m);
        else none_.dayTests(m);
    }
    void setStats(const uint32_t* t) {
        if (detailed_) Detailed::setStats(t);
    }
    std::tuple<unsigned, unsigned, unsigned> getStats() { return detailed_ ? Detailed::getStats() : none_.getStats(); }
    // NoTesting has no probabilities to update: the TPxxx flags change nothing
    void updateTestingProbs(const std::string& s) {
        if (detailed_) Detailed::updateTestingProbs(s);
    }
};

// RuleClosure or NoClosure, chosen at run time (--closurePolicy).  NoClosure
// reads no rules at all, so none of them acts, not even the ones that act
// with --enableClosures 0.
template <typename SimulationType>
class SelectableClosure : public RuleClosure<SimulationType> {
    using Rules = RuleClosure<SimulationType>;
    NoClosure<SimulationType> none_;
    bool rules_ = true;

public:
    using EngineHooks = SelectableClosure;
    void initializeArgs(const Options& o) {
        rules_ = o.closurePolicy != "none";
        if (rules_) Rules::initializeArgs(o);
        else none_.initializeArgs(o);
    }
    void init(const LocationTypeIds& lt, const std::vector<ClosureRuleRaw>& input, const std::string& header) {
        if (rules_) Rules::init(lt, input, header);
        else none_.init(lt, input, header);
    }
    void midnight(Timehandler t, unsigned dt, std::vector<unsigned>& stats) {
        if (rules_) Rules::midnight(t, dt, stats);
        else none_.midnight(t, dt, stats);
    }
    void step(Timehandler t, unsigned dt) {
        if (rules_) Rules::step(t, dt);
        else none_.step(t, dt);
    }
};

// The reference's concrete binding (cmake/config/in/configTypes.h.in:10-16),
// with the movement, testing and closure policies selectable at run time.
using ConfiguredSimulation = Simulation<std::array<double, 2>, unsigned, DynamicPPState, BasicAgentMeta,
                                        SelectableMovement, BasicInfection, SelectableTesting, SelectableClosure>;

}  // namespace ps
