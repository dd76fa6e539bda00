// SPH<WCSPH>, SPH<PCISPH> and SPH<IISPH> forward steps for gfx950 in sorted
// (cell-major) particle order.
//
// Reference: SPH<Method>::forward_step (sph/sph.ixx:350-354), WCSPH::forward
// (sph/sph.cpp:214-226, kernels sph/wcsph.cu), PCISPH::forward
// (sph/sph.cpp:296-315, sph/pcisph.cu) and IISPH::forward (sph/sph.cpp:409-428,
// sph/iisph.cu). Each step reorders the particles by cell once and fuses every
// per-particle chain into the neighbour pass that produces its input:
//
//   WCSPH          masks + density + Tait pressure -> rho, p, p / rho^2
//                  pressure + artificial viscosity + surface + external +
//                  integrate -> next state
//   PCISPH/IISPH   masks + density; non-pressure + first predict -> x*
//                  per iteration  A: rho* at x* (skin mask) + pressure update
//                                 B: pressure acceleration + predict -> x*
//                                    (the last one writes the next state)
//
// PCISPH and IISPH differ only in the volume of the pressure update
// (V = m / rho0 and V = m / rho). Sums run in the reference order over the
// neighbour masks, so results equal the reference expression by expression
// (the Tait pressure goes through the platform's powf).
#include <cmath>

#include "sph.hpp"
#include "sph_kernels.hpp"

namespace phx {
namespace {

struct WcsphForceArgs {
    uint32_t n;
    KernelConstants kc;
    float dt;
    float diameter;
    SortedGrid grid;
    Box box;
    Float3 gravity;
    const float4* xm;   // position + mass
    const float4* vmu;  // velocity + viscosity
    const float4* aux;  // density, p / rho^2, speed of sound, surface tension
    CVec u;
    const uint16_t* exact;
    const uint32_t* perm;
    Vec next_x, next_v;
    uint8_t* collisions;  // optional (recorded step): box-collision bits of the integration
    BoundaryGrid boundary;          // offsets null: no boundary samples
    const float* rest_density;      // rho0, for the boundary terms
    const float* boundary_tension;  // WCSPH boundary_surface_tension, for the boundary cohesion
    const uint8_t* crowded;         // per particle: walks the full stencil
    const uint32_t* cell;           // MaskDensityArgs::cell
    const uint16_t* exact_samples;  // MaskDensityArgs::exact_samples
};

// The sums of WCSPH::forward (sph.cpp:219-222), external_forward_kernel
// (wcsph.cu:86-90) and integrate_forward_kernel (common.cu:302-320) from
// particle i's pressure, viscosity and surface accelerations.
__device__ __forceinline__ void finish_wcsph(const WcsphForceArgs& a, uint32_t i, Float3 p, Float3 vel, Float3 ap,
                                             Float3 av, Float3 as) {
    Float3 total = add(ap, av);
    total = add(total, as);
    total = add(total, add(a.gravity, load(a.u, i)));
    Float3 nx, nv;
    predict_clamped(a.box, a.dt, p, vel, total, nx, nv);
    if (a.collisions != nullptr) a.collisions[i] = static_cast<uint8_t>(predict_collisions(a.box, a.dt, p, vel, total));
    const uint32_t j = a.perm[i];
    store(a.next_x, j, nx);
    store(a.next_v, j, nv);
}

// pressure_forward_kernel (common.cu:165-194), viscosity_forward_kernel
// (wcsph.cu:136-174), surface_forward_kernel (wcsph.cu:306-339) as three
// accumulators over one neighbour walk, then finish_wcsph. Always in groups:
// the pair terms are long enough that four lanes beat one at any size
// (16,000 particles 113 -> 63 us a step, 1,048,576: 614 -> 482 us, this pass
// 325 -> 213 us).
// With kSamples a boundary sample b, after each cell's particles, adds the pressure term
// grad W (-rho0_i V_b p_i / rho_i^2), on approach the artificial viscosity
// with nu = mu_i h c_i / rho_i and mass rho0_i V_b, and within h the cohesion
// -sigma_b,i rho0_i V_b W / m_i d (wcsph.cu:160-170, 326-335).
template <int G, bool kSamples>
__global__ void __launch_bounds__(kGroupBlock) wcsph_force_kernel(WcsphForceArgs a) {
    constexpr uint32_t kParticles = kGroupParticles<G>;
    constexpr int kSums = 9;
    __shared__ GroupLds<G> lds;
    const uint32_t base = xcd_block() * kParticles;
    const uint32_t i = base + threadIdx.x % kParticles;
    uint32_t center = 0u;
    bool listed = false;
    if (i < a.n) {
        center = a.cell[i];
        listed = a.crowded[i] == 0u;
    }
    const uint32_t w = base + threadIdx.x / G;
    const bool active = w < a.n;
    const uint32_t own_index = active ? w : 0u;
    const float h = a.kc.h;
    const float4 self = a.xm[own_index];
    const Float3 p = xyz(self);
    const float4 vm = a.vmu[own_index];
    const Float3 vel = xyz(vm);
    const float4 own = a.aux[own_index];
    const float rest = kSamples ? a.rest_density[own_index] : 0.0F;
    const float tension = kSamples ? a.boundary_tension[own_index] : 0.0F;
    const float softening = 0.01F * h * h;
    const float contact_weight = cubic_value(pair_distance(Float3{a.diameter, 0.0F, 0.0F}), a.kc);
    float sum[kSums] = {0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F};
    struct Record {
        float4 q, v, aux;
    };
    auto fetch = [&](uint32_t entry) {
        if constexpr (kSamples) {
            if ((entry & kSampleEntry) != 0u) {
                const uint32_t b = entry & ~kSampleEntry;
                return Record{a.boundary.x[b], a.boundary.v[b], float4{}};
            }
        }
        return Record{a.xm[entry], a.vmu[entry], a.aux[entry]};
    };
    auto put = [](float* terms, Float3 v) {
        terms[0] = v.x;
        terms[1] = v.y;
        terms[2] = v.z;
    };
    auto pair = [&](const Record& r, uint32_t entry, float (&terms)[kSums]) {
        const bool sample = kSamples && (entry & kSampleEntry) != 0u;
        const Float3 d = sub(p, xyz(r.q));
        const float dist = pair_distance(d);
        const Float3 gradient = scale(d, cubic_gradient_factor(dist, a.kc));
        put(terms, scale(gradient, sample ? -rest * r.q.w * own.y : -r.q.w * (own.y + r.aux.y)));
        const float compression = dot(sub(vel, xyz(r.v)), d);
        if (!(compression >= 0.0F)) {
            const float alpha = 0.5F * (vm.w + r.v.w);
            const float speed = 0.5F * (own.z + r.aux.z);
            const float nu = sample ? vm.w * h * own.z / own.x : 2.0F * alpha * h * speed / (own.x + r.aux.x);
            const float pi_value = -nu * compression / (dot(d, d) + softening);
            put(terms + 3, scale(gradient, sample ? -rest * r.q.w * pi_value : -r.q.w * pi_value));
        }
        if (!(dist >= h)) {
            const float weight = dist > a.diameter ? cubic_value(dist, a.kc) : contact_weight;
            const float factor = sample ? -tension * rest * r.q.w * weight / self.w : -own.w * r.q.w * weight / self.w;
            put(terms + 6, scale(d, factor));
        }
    };
    auto fold = [&](const float (&terms)[kSums]) { group_add<G, kSums>(sum, terms); };
    group_expand<G, kSamples>(
        lds,
        [&](auto& bits, auto& first) {
            if (listed) stored_slots<G, true>(a.exact, a.grid, a.grid.offsets, a.n, i, center, bits, first);
        },
        [&](auto& bits, auto& first) {
            if (listed) stored_slots<G, false>(a.exact_samples, a.grid, a.boundary.offsets, a.n, i, center, bits, first);
        },
        [&](const uint32_t* row, uint32_t count) {
            if (active) group_walk_list<G, kSums>(row, count, w, fetch, pair, fold);
        });
    if (!active) return;
    if (a.crowded[w] != 0u) {
        int cx, cy, cz;
        cell_coordinates(a.grid, a.cell[w], cx, cy, cz);
        group_walk_stencil<G, kSums>(
            a.grid, kSamples ? a.boundary.offsets : nullptr, cx, cy, cz, w, w, group_row(lds),
            [&](uint32_t entry) {
                const bool sample = kSamples && (entry & kSampleEntry) != 0u;
                return within_support(a.kc, p, xyz(sample ? a.boundary.x[entry & ~kSampleEntry] : a.xm[entry]));
            },
            fetch, pair, fold);
    }
    if (threadIdx.x % G == 0u)
        finish_wcsph(a, w, p, vel, Float3{sum[0], sum[1], sum[2]}, Float3{sum[3], sum[4], sum[5]},
                     Float3{sum[6], sum[7], sum[8]});
}

}  // namespace

const char* sph_pass_name(int pass) {
    static const char* names[kSphPassCount] = {"grid", "mask_density", "force_init", "projection", "force",
                                               "forces"};
    return pass >= 0 && pass < kSphPassCount ? names[pass] : "unknown";
}

double sph_pass_bytes(phx_sph_method method, int pass, uint32_t particles, uint32_t cells) {
    const double offsets = particles > 0 ? 4.0 * (static_cast<double>(cells) + 1.0) / particles : 0.0;
    const bool wcsph = method == PHX_SPH_WCSPH;
    switch (pass) {
        case kSphGrid:  // x, v, u (36) + m, rho0, mu and the method's per-particle parameters, read and written
                        // in cell order, + the permutation (4)
            return 2.0 * (36.0 + (wcsph ? 24.0 : 16.0)) + 4.0 + 2.0 * offsets;
        case kSphDensity:  // x, m in; rho out (WCSPH: + rho0, c, gamma, sigma in; p, p / rho^2 out)
            return wcsph ? 32.0 + 12.0 + offsets : 16.0 + 4.0 + offsets;
        case kSphForceInit:  // x, v, u, m, mu, rho in; a_np, x* out
            return 48.0 + 24.0 + offsets;
        case kSphProjection:  // x, x*, m, rho, rho0, relaxation, p in; p, p / rho^2 out
            return 44.0 + 8.0 + offsets;
        case kSphForce:  // x, v, m, p / rho^2, a_np in; x* out
            return 44.0 + 12.0 + offsets;
        case kSphForces:  // x, v, u, m, mu, rho, p / rho^2, c, sigma in; next x, v out
            return 60.0 + 24.0 + offsets;
        default:
            return 0.0;
    }
}

void SphCache::allocate(uint32_t n, uint32_t cells) {
    neighborhood.allocate(n, cells);
    densities.resize(n);
    pressures.resize(n);
    if (method != PHX_SPH_WCSPH) non_pressure.resize(n);
}

SphSolver::SphSolver(const phx_domain_configuration* domain, const phx_sph_configuration* configuration,
                     phx_execution_mode mode, hipStream_t stream)
    : domain_(make_domain(domain)), mode_(mode), stream_(stream) {
    require(configuration != nullptr, PHX_ERROR_INVALID_ARGUMENT, "null SPH configuration");

    config_ = *configuration;
    require(config_.method == PHX_SPH_WCSPH || config_.method == PHX_SPH_PCISPH || config_.method == PHX_SPH_IISPH,
            PHX_ERROR_INVALID_ARGUMENT, "unknown SPH method");
    require(mode == PHX_MODE_FORWARD || mode == PHX_MODE_DIFFERENTIABLE, PHX_ERROR_INVALID_ARGUMENT,
            "unknown execution mode");
    boundary_.upload(domain_.config);
    domain_.config.boundary_particles = nullptr;  // the caller's host array is not kept
    const float tolerance = config_.density_error_tolerance;
    require(tolerance >= 0.0F && std::isfinite(tolerance), PHX_ERROR_INVALID_ARGUMENT,
            "density_error_tolerance must be finite and non-negative");
    if (config_.method != PHX_SPH_WCSPH) {
        require(config_.checkpoint_interval > 0u, PHX_ERROR_INVALID_ARGUMENT, "checkpoint_interval must be positive");
        require(config_.pressure_iterations < 4096u, PHX_ERROR_INVALID_ARGUMENT, "too many pressure iterations");
        require(tolerance == 0.0F || mode == PHX_MODE_FORWARD, PHX_ERROR_UNSUPPORTED,
                "tolerance mode is supported in forward mode only");
        require(tolerance == 0.0F || (config_.max_iterations >= 1u && config_.max_iterations < 2048u),
                PHX_ERROR_INVALID_ARGUMENT, "tolerance mode needs 1 <= max_iterations < 2048");
    } else {
        require(tolerance == 0.0F, PHX_ERROR_INVALID_ARGUMENT, "tolerance mode applies to PCISPH and IISPH");
        config_.pressure_iterations = 0u;
    }
    gradient_norm_ = reference_gradient_norm(domain_.config);
    constants_ = kernel_constants(domain_.config.support_radius);
    const uint32_t n = domain_.config.particle_count;
    for (DeviceBuffer<float4>* b : {&vmu_, &aux_}) b->resize(n);
    for (DeviceBuffer<float4>* b : {&xm_, &xs_}) b->resize(n + static_cast<size_t>(kScanPadding));
    u_.resize(n);
    for (DeviceBuffer<float>* b : {&rho0_, &relax_, &tait_, &t_}) b->resize(n);
    if (boundary_.count() > 0u && config_.method == PHX_SPH_WCSPH) btension_.resize(n);
    // one displacement slot per predicting pass
    const uint32_t predictions = (tolerance > 0.0F ? config_.max_iterations : config_.pressure_iterations) + 1u;
    masks_.allocate(n, predictions, domain_.config.support_radius);
    if (boundary_.count() > 0u) {
        exact_samples_.resize(static_cast<size_t>(kStencil) * n);
        skin_samples_.resize(static_cast<size_t>(kStencil) * n);
    }
    if (mode == PHX_MODE_FORWARD && config_.method != PHX_SPH_WCSPH) {
        xt_.resize(n);
        mass_state_.resize(2u);
        fill_u32(stream_, mass_state_.data(), 2u, 0u);
        for (DeviceBuffer<float>* b : {&moved_, &moved_sorted_}) b->resize(n);
        cell_bound_.resize(domain_.cells);
        taint_.resize(domain_.cells);
        fill_u32(stream_, taint_.data(), domain_.cells, 0u);
    }
    if (tolerance > 0.0F) {
        tol_partials_.resize(static_cast<size_t>(pass_blocks(n, pass_group(n, boundary_.count() > 0u))) * kWaves);  // one per projection wave
        tol_done_.resize(1u);
        tol_host_.resize(2u * sizeof(uint32_t));
        for (hipEvent_t& e : tol_events_) PHX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    if (mode == PHX_MODE_DIFFERENTIABLE && config_.method != PHX_SPH_WCSPH) {
        // PCISPH::forward (sph.cpp:295-309) and IISPH::forward (sph.cpp:408-421)
        // are the DFSPH step with nd = 0, no warm start and their relaxation in
        // the density phase: the divergence phase then adds a zero
        // acceleration, and the pressure update's volume is m / rho0 (PCISPH)
        // or m / rho (IISPH)
        phx_dfsph_configuration dc{};
        dc.divergence_iterations = 0u;
        dc.density_iterations = config_.pressure_iterations;
        dc.checkpoint_interval = config_.checkpoint_interval;
        dc.pressure_warm_start = 0u;
        dc.exact_no_slip_adjoint = config_.exact_no_slip_adjoint;
        engine_ = std::make_unique<DfsphSolver>(domain, &dc, PHX_MODE_DIFFERENTIABLE, stream);
        engine_->set_volume_rest_density(config_.method == PHX_SPH_PCISPH);
        for (auto& b : engine_warm_) b.resize(n);
    }
}

SphSolver::~SphSolver() {
    for (hipEvent_t e : tol_events_)
        if (e != nullptr) (void)hipEventDestroy(e);
}

void SphSolver::require_derivatives(const SphCache& cache) const {
    require(mode_ == PHX_MODE_DIFFERENTIABLE, PHX_ERROR_UNSUPPORTED,
            "derivatives need a solver created in differentiable mode");
    const bool recorded = config_.method == PHX_SPH_WCSPH ? cache.wcsph != nullptr && cache.wcsph->recorded
                                                          : cache.record != nullptr && cache.record->recorded;
    require(recorded && cache.method == config_.method, PHX_ERROR_INVALID_ARGUMENT,
            "the step cache holds no step recorded by this solver");
    require(cache.grid().particles == domain_.config.particle_count, PHX_ERROR_INVALID_ARGUMENT,
            "the step cache belongs to another particle count");
}

void SphSolver::jvp_step(const SphCache& cache, const phx_sph_state_tangent& state_t,
                         const phx_control_tangent& control_t, const phx_sph_parameter_tangent& parameter_t,
                         phx_sph_state_tangent& next_t) {
    require_derivatives(cache);
    if (config_.method == PHX_SPH_WCSPH) {
        wcsph_jvp_step(cache, state_t, control_t, parameter_t, next_t);
        return;
    }
    const bool iisph = config_.method == PHX_SPH_IISPH;
    phx_sph_dfsph_state_tangent st{state_t.particles, {nullptr, nullptr}};
    phx_sph_dfsph_state_tangent nt{next_t.particles, {nullptr, nullptr}};
    phx_sph_dfsph_parameter_tangent pt{
        parameter_t.particles,
        {nullptr, iisph ? parameter_t.method.jacobi_relaxation : parameter_t.method.pressure_relaxation}};
    engine_->jvp_step(*cache.record, st, control_t, pt, nt);
}

void SphSolver::vjp_step(const SphCache& cache, const phx_sph_state_adjoint& next_a,
                         phx_sph_state_adjoint& previous_a, phx_control_adjoint& control_a,
                         phx_sph_parameter_adjoint& parameter_a) {
    require_derivatives(cache);
    if (config_.method == PHX_SPH_WCSPH) {
        wcsph_vjp_step(cache, next_a, previous_a, control_a, parameter_a);
        return;
    }
    const bool iisph = config_.method == PHX_SPH_IISPH;
    phx_sph_dfsph_state_adjoint na{next_a.particles, {nullptr, nullptr}};
    phx_sph_dfsph_state_adjoint pa{previous_a.particles, {nullptr, nullptr}};
    phx_sph_dfsph_parameter_adjoint pp{
        parameter_a.particles,
        {nullptr, iisph ? parameter_a.method.jacobi_relaxation : parameter_a.method.pressure_relaxation}};
    engine_->vjp_step(*cache.record, na, pa, control_a, pp);
}

void SphSolver::forward_step(const phx_sph_state& state, const phx_control& control,
                             const phx_sph_parameters& parameters, phx_sph_state& next, SphCache& cache) {
    const uint32_t n = domain_.config.particle_count;
    if (n == 0) {
        next.particles.step_index = state.particles.step_index + 1u;
        return;
    }
    require_vec(state.particles.positions, "state positions");
    require_vec(state.particles.velocities, "state velocities");
    require_vec(control.external_accelerations, "control");
    require_vec(next.particles.positions, "next positions");
    require_vec(next.particles.velocities, "next velocities");
    const auto& pp = parameters.particles;
    require(pp.masses && pp.rest_densities && pp.viscosities, PHX_ERROR_INVALID_ARGUMENT, "null particle parameters");
    cache.method = config_.method;
    if (engine_) {
        const float* relaxation = config_.method == PHX_SPH_IISPH ? parameters.method.jacobi_relaxation
                                                                  : parameters.method.pressure_relaxation;
        require(relaxation != nullptr, PHX_ERROR_INVALID_ARGUMENT,
                config_.method == PHX_SPH_IISPH ? "null IISPH jacobi_relaxation" : "null PCISPH pressure_relaxation");
        if (!cache.record) cache.record = std::make_unique<DfsphCache>();
        cache.stream = stream_;
        phx_sph_dfsph_state s{state.particles, {nullptr, nullptr}};
        phx_sph_dfsph_state nx{next.particles, {engine_warm_[0].data(), engine_warm_[1].data()}};
        phx_sph_dfsph_parameters p{parameters.particles, {relaxation, relaxation}};
        engine_->forward_step(s, control, p, nx, *cache.record);
        next.particles.step_index = nx.particles.step_index;
        return;
    }
    cache.record.reset();
    cache.allocate(n, domain_.cells);
    if (config_.method == PHX_SPH_WCSPH) {
        forward_wcsph(state, control, parameters, next, cache);
    } else {
        forward_pressure(state, control, parameters, next, cache);
    }
    next.particles.step_index = state.particles.step_index + 1u;
}

void SphSolver::forward_wcsph(const phx_sph_state& state, const phx_control& control,
                              const phx_sph_parameters& parameters, phx_sph_state& next, SphCache& cache) {
    const auto& c = domain_.config;
    const uint32_t n = c.particle_count;
    const uint64_t step = state.particles.step_index;
    const auto& pp = parameters.particles;
    const auto& mp = parameters.method;
    require(pp.surface_tensions && mp.speed_of_sound && mp.tait_exponent && mp.boundary_surface_tension,
            PHX_ERROR_INVALID_ARGUMENT, "null WCSPH parameters");
    // a recorded step keeps its sorted inputs, masks and collision bits in the cache
    const bool rec = mode_ == PHX_MODE_DIFFERENTIABLE;
    WcsphRecord* r = nullptr;
    if (rec) {
        if (!cache.wcsph) cache.wcsph = std::make_unique<WcsphRecord>();
        r = cache.wcsph.get();
        r->recorded = false;
        for (DeviceBuffer<float4>* b : {&r->vmu, &r->aux}) b->resize(n);
        r->xm.resize(n + static_cast<size_t>(kScanPadding));
        for (DeviceBuffer<float>* b : {&r->rho0, &r->tait}) b->resize(n);
        r->collisions.resize(n);
        r->exact.resize(static_cast<size_t>(kStencil) * n);
        r->crowded.resize(n);
        r->flags.resize(masks_.flag_count());
        if (boundary_.count() > 0u) r->btension.resize(n);
    }
    float4* xm = rec ? r->xm.data() : xm_.data();
    float4* vmu = rec ? r->vmu.data() : vmu_.data();
    float4* aux = rec ? r->aux.data() : aux_.data();
    float* rho0 = rec ? r->rho0.data() : rho0_.data();
    float* tait = rec ? r->tait.data() : tait_.data();
    uint16_t* exact = rec ? r->exact.data() : masks_.exact();
    uint8_t* crowded = rec ? r->crowded.data() : masks_.crowded();
    ChannelList gather;
    gather.add(cvec(state.particles.positions), xm);
    gather.add(pp.masses, xm, 3);
    gather.add(cvec(state.particles.velocities), vmu);
    gather.add(pp.viscosities, vmu, 3);
    gather.add(cvec(control.external_accelerations), u_.view());
    gather.add(pp.rest_densities, rho0);
    gather.add(mp.speed_of_sound, aux, 2);
    gather.add(pp.surface_tensions, aux, 3);
    gather.add(mp.tait_exponent, tait);
    const bool with_boundary = boundary_.count() > 0u;
    float* btension = rec && with_boundary ? r->btension.data() : btension_.data();
    if (with_boundary) gather.add(mp.boundary_surface_tension, btension);
    {
        PassScope scope(profiler_, stream_, kSphGrid);
        cache.neighborhood.build(stream_, domain_, step, cvec(state.particles.positions), nullptr, gather.get(),
                                 &boundary_);
        masks_.begin_step(stream_);
    }
    const SortedGrid grid = cache.neighborhood.grid();
    const BoundaryGrid boundary = cache.neighborhood.boundary();

    MaskDensityArgs ma{};
    ma.n = n;
    ma.kc = constants_;
    ma.t_skin = masks_.t_skin();
    ma.grid = grid;
    ma.boundary = boundary;
    ma.xm = xm;
    ma.exact = exact;
    ma.skin = masks_.skin_mask();
    ma.rho = cache.densities.data();
    ma.rest_density = rho0;
    ma.tait_exponent = tait;
    ma.pressures = cache.pressures.data();
    ma.aux = aux;
    ma.crowded = crowded;
    ma.cell = masks_.cells();
    ma.exact_samples = exact_samples_.data();
    ma.skin_samples = skin_samples_.data();
    launch_mask_density<true>(profiler_, stream_, ma, kSphDensity);

    WcsphForceArgs wa{};
    wa.n = n;
    wa.kc = constants_;
    wa.dt = c.time_step;
    wa.diameter = 2.0F * c.particle_radius;
    wa.grid = grid;
    wa.box = collision_box(c, step);
    wa.gravity = Float3{c.gravity.x, c.gravity.y, c.gravity.z};
    wa.xm = xm;
    wa.vmu = vmu;
    wa.aux = aux;
    wa.u = u_.cview();
    wa.exact = exact;
    wa.perm = cache.neighborhood.perm.data();
    wa.next_x = vec(next.particles.positions);
    wa.next_v = vec(next.particles.velocities);
    wa.collisions = rec ? r->collisions.data() : nullptr;
    wa.boundary = boundary;
    wa.rest_density = rho0;
    wa.boundary_tension = btension;
    wa.crowded = crowded;
    wa.cell = masks_.cells();
    wa.exact_samples = exact_samples_.data();
    {
        PassScope scope(profiler_, stream_, kSphForces);
        const int group = wide_group(n);
        with_group(group, with_boundary, [&](auto g, auto samples) {
            wcsph_force_kernel<g(), samples()><<<pass_blocks(n, group), kGroupBlock, 0, stream_>>>(wa);
        });
        PHX_LAUNCH_CHECK();
    }
    if (rec) {
        PHX_HIP(hipMemcpyAsync(r->flags.data(), masks_.flags(), sizeof(uint32_t) * masks_.flag_count(),
                               hipMemcpyDeviceToDevice, stream_));
        // the derivative passes walk the full stencil with samples
        if (with_boundary) fill_u32(stream_, r->flags.data() + kFlagOverflow, 1u, 1u);
        r->step_index = step;
        r->recorded = true;
    }
    masks_.end_step(stream_);
}

void SphSolver::forward_pressure(const phx_sph_state& state, const phx_control& control,
                                 const phx_sph_parameters& parameters, phx_sph_state& next, SphCache& cache) {
    const auto& c = domain_.config;
    const uint32_t n = c.particle_count;
    const uint64_t step = state.particles.step_index;
    const auto& pp = parameters.particles;
    const bool iisph = config_.method == PHX_SPH_IISPH;
    const float* relaxation = iisph ? parameters.method.jacobi_relaxation : parameters.method.pressure_relaxation;
    require(relaxation != nullptr, PHX_ERROR_INVALID_ARGUMENT,
            iisph ? "null IISPH jacobi_relaxation" : "null PCISPH pressure_relaxation");
    ChannelList gather;
    gather.add(cvec(state.particles.positions), xm_.data());
    gather.add(pp.masses, xm_.data(), 3);
    gather.add(cvec(state.particles.velocities), vmu_.data());
    gather.add(pp.viscosities, vmu_.data(), 3);
    gather.add(cvec(control.external_accelerations), u_.view());
    gather.add(pp.rest_densities, rho0_.data());
    gather.add(relaxation, relax_.data());
    const bool with_boundary = boundary_.count() > 0u;
    // per-cell skins (DfsphSolver::forward_step) from the previous step's displacements
    const bool cell_skins = have_moved_;
    if (cell_skins) gather.add(moved_.data(), moved_sorted_.data());
    const uint32_t predictions =
        (config_.density_error_tolerance > 0.0F ? config_.max_iterations : config_.pressure_iterations) + 1u;
    if (cell_skins && stamp_base_ > 0xFFFFFFFFu - predictions) {
        fill_u32(stream_, taint_.data(), domain_.cells, 0u);
        stamp_base_ = 1u;
    }
    {
        PassScope scope(profiler_, stream_, kSphGrid);
        cache.neighborhood.build(stream_, domain_, step, cvec(state.particles.positions), nullptr, gather.get(),
                                 &boundary_);
        masks_.begin_step(stream_);
        fill_f32(stream_, cache.pressures.data(), n, 0.0F);  // clear_iteration (sph.cpp:298)
        // the mask pass marks unequal masses with this step's stamp
        if (++mass_stamp_ == 0u) {
            fill_u32(stream_, mass_state_.data(), 1u, 0u);
            mass_stamp_ = 1u;
        }
        if (cell_skins) {
            const uint32_t cells = domain_.cells;
            cell_bound_kernel<<<blocks_for(cells, kBlock), kBlock, 0, stream_>>>(
                cells, cache.neighborhood.grid().offsets, moved_sorted_.data(), 1.2F, 0.01F * c.support_radius,
                cell_bound_.data());
            PHX_LAUNCH_CHECK();
        }
    }
    const SortedGrid grid = cache.neighborhood.grid();
    const BoundaryGrid boundary = cache.neighborhood.boundary();
    const int group = pass_group(n, with_boundary);
    const uint32_t blocks = pass_blocks(n, group);

    MaskDensityArgs ma{};
    ma.n = n;
    ma.kc = constants_;
    ma.t_skin = masks_.t_skin();
    ma.grid = grid;
    ma.boundary = boundary;
    ma.rest_density = rho0_.data();
    ma.xm = xm_.data();
    ma.exact = masks_.exact();
    ma.skin = masks_.skin_mask();
    ma.rho = cache.densities.data();
    ma.crowded = masks_.crowded();
    ma.cell = masks_.cells();
    ma.exact_samples = exact_samples_.data();
    ma.skin_samples = skin_samples_.data();
    if (cell_skins) ma.cell_bound = cell_bound_.data();
    ma.mass_state = mass_state_.data();
    ma.mass_stamp = mass_stamp_;
    launch_mask_density<false>(profiler_, stream_, ma, kSphDensity);

    ForceArgs fa{};
    fa.n = n;
    fa.kc = constants_;
    fa.dt = c.time_step;
    fa.grid = grid;
    fa.box = collision_box(c, step);
    fa.gravity = Float3{c.gravity.x, c.gravity.y, c.gravity.z};
    fa.xm = xm_.data();
    fa.vmu = vmu_.data();
    fa.u = u_.cview();
    fa.rho = cache.densities.data();
    fa.t1 = t_.data();
    fa.exact = masks_.exact();
    fa.flags = masks_.flags();
    fa.anp = cache.non_pressure.data();
    fa.xs = xs_.data();
    fa.perm = cache.neighborhood.perm.data();
    fa.next_x = vec(next.particles.positions);
    fa.next_v = vec(next.particles.velocities);
    fa.boundary = boundary;
    fa.rest_density = rho0_.data();
    fa.crowded = masks_.crowded();
    fa.cell = masks_.cells();
    fa.moved_out = moved_.data();
    fa.xt1 = xt_.data();
    fa.mass_state = mass_state_.data();
    fa.mass_stamp = mass_stamp_;
    fa.exact_samples = exact_samples_.data();
    if (cell_skins) {
        fa.cell_bound = cell_bound_.data();
        fa.taint = taint_.data();
    }

    ProjectionArgs pa{};
    pa.n = n;
    pa.kc = constants_;
    pa.dt = c.time_step;
    pa.gradient_norm = gradient_norm_;
    pa.limit2 = masks_.limit2();
    pa.grid = grid;
    pa.xm = xm_.data();
    pa.xs = xs_.data();
    pa.skin = masks_.skin_mask();
    pa.flags = masks_.flags();
    pa.rho = cache.densities.data();
    pa.volume_density = iisph ? cache.densities.data() : rho0_.data();
    pa.target = rho0_.data();
    pa.relaxation = relax_.data();
    pa.p_prev = cache.pressures.data();
    pa.p = cache.pressures.data();
    pa.t = t_.data();
    pa.boundary = boundary;
    pa.rest_density = rho0_.data();
    pa.crowded = masks_.crowded();
    pa.cell = masks_.cells();
    pa.skin_samples = skin_samples_.data();
    pa.xt_out = xt_.data();
    if (cell_skins) pa.taint = taint_.data();
    // the stamps of this step's predictions: stamp_base_ + slot
    auto set_force_slot = [&](uint32_t slot) {
        fa.slot = slot;
        fa.stamp = stamp_base_ + slot;
    };
    auto set_projection_slot = [&](uint32_t slot) {
        pa.slot = slot;
        pa.stamp = stamp_base_ + slot;
    };
    auto end_step = [&] {
        masks_.end_step(stream_);
        if (cell_skins) stamp_base_ += predictions;
        have_moved_ = true;  // the final pass wrote every particle's displacement
    };

    if (config_.density_error_tolerance > 0.0F) {
        // Tolerance mode: iterate until the projection's mean compression
        // error is within the tolerance (or max_iterations); the force pass
        // of that iteration writes the state. As DfsphSolver's tolerance
        // mode, the host reads an iteration's done word while its force
        // pass runs, then launches the next iteration.
        const uint32_t max_it = config_.max_iterations;
        const double tolerance = static_cast<double>(config_.density_error_tolerance);
        uint32_t* done = tol_done_.data();
        const volatile uint32_t* host = static_cast<uint32_t*>(tol_host_.data());
        auto* host_device = static_cast<uint32_t*>(tol_host_.device());
        fill_u32(stream_, done, 1u, 0u);
        set_force_slot(0u);
        fa.final_step = 0u;
        launch_force<true, kInitPredict>(profiler_, stream_, group, fa, kSphForceInit);
        auto launch_iteration = [&](uint32_t it) {
            set_projection_slot(it - 1u);  // the prediction of the previous pass
            pa.cv = Convergence{tol_partials_.data(), done, rho0_.data()};
            launch_projection(profiler_, stream_, group, pa, kSphProjection, kProjectDensity);
            converge_kernel<<<1, kConvergeBlock, 0, stream_>>>(tol_partials_.data(), blocks * kWaves, n, tolerance,
                                                               it, max_it, done, host_device + (it & 1u));
            PHX_HIP(hipGetLastError());
            PHX_HIP(hipEventRecord(tol_events_[it & 1u], stream_));
            set_force_slot(it);
            fa.done = done;
            fa.iteration = it;
            fa.final_step = 0u;
            launch_force<false, kDivPredict>(profiler_, stream_, group, fa, kSphForce);
        };
        launch_iteration(1u);
        uint32_t it = 1u;
        for (;; ++it) {
            // the force pass of this iteration runs while the host reads its done word
            PHX_HIP(hipEventSynchronize(tol_events_[it & 1u]));
            // the projection of iteration max_it always ends the step
            if (host[it & 1u] != 0u || it >= max_it) break;
            launch_iteration(it + 1u);
        }
        last_iterations_ = it;
        pa.cv = Convergence{};
        fa.done = nullptr;
        end_step();
        return;
    }
    const uint32_t iterations = config_.pressure_iterations;
    last_iterations_ = iterations;
    uint32_t slot = 0;  // displacement slot written by the latest predicting pass
    set_force_slot(slot);
    fa.final_step = iterations == 0u ? 1u : 0u;
    launch_force<true, kInitPredict>(profiler_, stream_, group, fa, kSphForceInit);
    for (uint32_t it = 1; it <= iterations; ++it) {  // sph.cpp:300-307 / 413-420
        set_projection_slot(slot);
        launch_projection(profiler_, stream_, group, pa, kSphProjection, kProjectDensity);
        set_force_slot(++slot);
        fa.final_step = it == iterations ? 1u : 0u;
        launch_force<false, kDivPredict>(profiler_, stream_, group, fa, kSphForce);
    }
    end_step();
}

}  // namespace phx
