#include "tlookup.hpp"

#include <cstring>

#include "../../include/zkllm_hip.h"
#include "../csrc/field.hpp"

#define ZKC(call) zk_check((call), #call)

static const Fr_t kOne{{1, 0, 0, 0, 0, 0, 0, 0}};
// 1/2 mod r (tlookup.cu:179-180)
static const Fr_t TWO_INV{{2147483649u, 2147483647u, 2147429887u, 2849952257u, 80800770u, 429714436u, 2496577188u, 972477353u}};

tLookup::tLookup(const FrTensor& table) : table(table) {}
tLookup::tLookup(FrTensor&& table) : table(std::move(table)) {}

// multiplicities of a table's N entries from positions
static FrTensor counts_to_m(const void* idx, uint D, uint N) {
    FrTensor m(N);
    ZKC(zk_lookup_multiplicities(m.gpu_data, nullptr, idx, nullptr, nullptr, 0, N, D, N, 0, nullptr));
    return m;
}
// the same from queries in int32 form: positions value - low formed by the counting passes themselves
static FrTensor counts_to_m_i32(const void* vals_i32, int low, uint len, uint D, uint N) {
    FrTensor m(N);
    ZKC(zk_lookup_multiplicities(m.gpu_data, nullptr, nullptr, vals_i32, nullptr, low, len, D, N, 0, nullptr));
    return m;
}
// and from the queries themselves
static FrTensor counts_to_m(const FrTensor& vals, int low, uint len, uint N, bool inside = false) {
    const void* h = vals.kept_ints();
    FrTensor m(N);
    ZKC(zk_lookup_multiplicities(m.gpu_data, nullptr, nullptr, h ? zk_fr_fold_prepared_ints(h) : nullptr, vals.gpu_data, low, len, vals.size, N, inside, nullptr));
    return m;
}
LookupOpened::~LookupOpened() { if (handle) (void)zk_lookup_open_drop(handle); }
CountedQueries::~CountedQueries() { if (check) (void)zk_lookup_multiplicities_end(check); }
void CountedQueries::settle() {
    void* c = check;
    check = nullptr;
    if (c) ZKC(zk_lookup_multiplicities_end(c));
}

FrTensor tLookup::prep(const uint* indices, const uint D) { return counts_to_m(indices, D, table.size); }

static FrTensor make_range_table(int low, uint len) {
    FrTensor t(1u << ceilLog2(len));
    ZKC(zk_range_table(t.gpu_data, low, len, t.size, nullptr));
    return t;
}
tLookupRange::tLookupRange(int low, uint len) : tLookup(make_range_table(low, len)), low(low), len(len) {}

FrTensor tLookupRange::prep(const int* vals, const uint D) { return counts_to_m_i32(vals, low, len, D, table.size); }
FrTensor tLookupRange::prep(const FrTensor& vals) { return counts_to_m(vals, low, len, table.size); }
FrTensor tLookupRange::prep_inside(const FrTensor& vals) { return counts_to_m(vals, low, len, table.size, true); }

// mapped values padded by repeating the last one (tlookup.cu:435-444)
static FrTensor make_mapped(uint len, const FrTensor& mvals) {
    if (mvals.size != len) throw std::runtime_error("mvals.size != len");
    FrTensor out(1u << ceilLog2(len));
    ZKC(zk_fr_pad_from(out.gpu_data, mvals.gpu_data, mvals.size, out.size, mvals.gpu_data + (mvals.size - 1), nullptr));
    return out;
}
tLookupRangeMapping::tLookupRangeMapping(int low, uint len, const FrTensor& mvals) : tLookupRangeMapping(low, len, mvals, queued) {
    (void)mapped_vals.kept_ints();          // waits
}
tLookupRangeMapping::tLookupRangeMapping(int low, uint len, const FrTensor& mvals, Queued) : tLookupRange(low, len), mapped_vals(make_mapped(len, mvals)) {
    mapped_vals.keep_for_folds_queued();          // examined once: outputs of operator() carry an int32 form when these are 32-bit integers
}

pair<FrTensor, FrTensor> tLookupRangeMapping::operator()(const int* vals, const uint D) {
    DevBuf idx(sizeof(uint) * (size_t)D);
    FrTensor m(table.size);
    ZKC(zk_lookup_multiplicities(m.gpu_data, idx.p, nullptr, vals, nullptr, low, len, D, table.size, 0, nullptr));
    FrTensor y(D);
    ZKC(zk_fr_gather(y.gpu_data, mapped_vals.gpu_data, idx.p, D, nullptr));
    ZKC(zk_sync(nullptr));
    return {std::move(y), std::move(m)};
}
pair<FrTensor, FrTensor> tLookupRangeMapping::operator()(const FrTensor& vals) { return map(vals, nullptr); }
pair<FrTensor, FrTensor> tLookupRangeMapping::map(const FrTensor& vals, const FrTensor* unwritten) {
    auto p = map_queued(vals, unwritten);
    ZKC(zk_sync(nullptr));
    return p;
}
pair<FrTensor, FrTensor> tLookupRangeMapping::map_queued(const FrTensor& vals, const FrTensor* unwritten) {
    CountedQueries c;
    // queries and mapped values in int32 form: nothing below needs the array of table positions
    count(c, vals, !(vals.kept_ints() && mapped_vals.kept_ints()), true);
    FrTensor y = gather(vals, c, unwritten);
    return {std::move(y), std::move(*c.m)};
}
// wait: the range check is settled here (an attention head of 2 x 128 tokens takes 20 us less so than by settle() in the next line)
void tLookupRangeMapping::count(CountedQueries& c, const FrTensor& vals, bool positions, bool wait) {
    if (positions) c.idx.reset(new DevBuf(sizeof(uint) * (size_t)vals.size));
    const void* h = vals.kept_ints();
    const void* ints = h ? zk_fr_fold_prepared_ints(h) : nullptr;
    void* idx = positions ? c.idx->p : nullptr;
    c.m.reset(new FrTensor(table.size));
    if (wait) ZKC(zk_lookup_multiplicities(c.m->gpu_data, idx, nullptr, ints, vals.gpu_data, low, len, vals.size, table.size, 0, nullptr));
    else ZKC(zk_lookup_multiplicities_begin(&c.check, c.m->gpu_data, idx, nullptr, ints, vals.gpu_data, low, len, vals.size, table.size, nullptr));
}
// the outputs of counted queries
FrTensor tLookupRangeMapping::gather(const FrTensor& vals, const CountedQueries& c, const FrTensor* unwritten) {
    const bool ints_only_out = unwritten && unwritten->size == vals.size && mapped_vals.kept_ints() && vals.kept_ints();
    FrTensor y = ints_only_out ? FrTensor::view(*unwritten) : FrTensor(vals.size);
    // mapped values that are 32-bit integers: the outputs get their int32 form with them
    if (const void* th = mapped_vals.kept_ints(); th && vals.kept_ints()) {
        // queries with an int32 form: gathered by them, and the outputs' form remembers it (the proof's first round then trusts them)
        y.ints_for_producer();
        ZKC(zk_fr_gather_by_queries_ints(ints_only_out ? nullptr : y.gpu_data, const_cast<void*>(y.kept_ints()), vals.kept_ints(), low, th, vals.size, nullptr));
    } else if (th) ZKC(zk_fr_gather_ints(y.gpu_data, y.ints_for_producer(), mapped_vals.gpu_data, th, c.idx->p, vals.size, nullptr));
    else ZKC(zk_fr_gather(y.gpu_data, mapped_vals.gpu_data, c.idx->p, vals.size, nullptr));
    return y;
}

static void drop_lookup_job(void* h, size_t rounds) {
    if (!h) return;
    std::vector<Fr_t> sums(rounds * 11 + 1);
    Fr_t bm;
    (void)zk_lookup_prove_end(h, bm.val, sums[0].val);
}
LookupPending::~LookupPending() { drop_lookup_job(handle, u.size()); }
LookupPending& LookupPending::operator=(LookupPending&& o) noexcept {
    if (this != &o) {
        drop_lookup_job(handle, u.size());
        handle = o.handle; o.handle = nullptr;
        keep = std::move(o.keep);
        alpha = o.alpha; beta = o.beta;
        u = std::move(o.u); v = std::move(o.v);
        D = o.D; N = o.N;
    }
    return *this;
}

// tLookup_phase1 / tLookup_phase2 (tlookup.cu:184-320).  The device side -- inverses, <B, m>, eq table and every round --
// is one job that runs beside the caller; the host side turns each round's sums into its polynomial, checks it and
// derives the next claim.
// S_out / r given: S0 holds the input queries of a mapping table, the combined query S0 + r * S_out is formed on the device
static LookupPending sumcheck_begin(const FrTensor& S0, const FrTensor& T0, const FrTensor& m0, const Fr_t& alpha0, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v,
                                    const FrTensor* hint, int low, const FrTensor* S_out, const Fr_t* r, const void* mapped_ints = nullptr, LookupOpened* opened = nullptr, bool queries_ready = false, bool at_once = false);
LookupPending tLookup_sumcheck_begin(const FrTensor& S0, const FrTensor& T0, const FrTensor& m0, const Fr_t& alpha0, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v,
                                     const FrTensor* hint, int low) {
    return sumcheck_begin(S0, T0, m0, alpha0, beta, u, v, hint, low, nullptr, nullptr);
}
// mapped_ints: the int32 form of the mapping table's (padded) mapped values, when it keeps one
static LookupPending sumcheck_begin(const FrTensor& S0, const FrTensor& T0, const FrTensor& m0, const Fr_t& alpha0, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v,
                                    const FrTensor* hint, int low, const FrTensor* S_out, const Fr_t* r, const void* mapped_ints, LookupOpened* opened, bool queries_ready, bool at_once) {
    const uint D = S0.size, N = m0.size;
    if (S_out && S_out->size != D) throw std::runtime_error("lookup: input and output queries differ in size");
    if (m0.size != T0.size) throw std::runtime_error("m.size != table.size");
    if (D != (1u << ceilLog2(D)) || N != (1u << ceilLog2(N)) || D % N != 0) throw std::runtime_error("D or N is not power of 2, or D is not divisible by N");
    if (u.size() != ceilLog2(D)) throw std::runtime_error("u.size() != ceilLog2(D)");
    if (v.size() != ceilLog2(D)) throw std::runtime_error("v.size() != ceilLog2(D)");
    LookupPending p;
    p.alpha = alpha0; p.beta = beta; p.u = u; p.v = v; p.D = D; p.N = N;
    const uint k = (uint)u.size();
    if (k == 0) return p;
    const uint n1 = ceilLog2(D / N);
    // fold challenges in round order: v1 = v[0..n1) consumed from its back, then v2 = v[n1..k) from its back
    std::vector<Fr_t> vs(k);
    for (uint r = 0; r < k; ++r) vs[r] = r >= n1 ? v[k - 1 - (r - n1)] : v[n1 - 1 - r];
    if (hint && hint->size != D) throw std::runtime_error("lookup hint must have one entry per query");
    // queries that keep an int32 form (the digit planes of a softmax, the outputs of a mapping table) are read from it
    const void *qi = S0.kept_ints(), *oi = S_out ? S_out->kept_ints() : nullptr;
    if (opened) {          // hint: the queries, or the mapped queries
        ZKC(zk_lookup_prove_begin_opened(&p.handle, opened->handle, S0.gpu_data, qi, S_out ? S_out->gpu_data : nullptr, oi, mapped_ints, r ? r->val : nullptr, T0.gpu_data, m0.gpu_data, low,
                                         beta.val, u[0].val, vs[0].val, D, N, (int)k, queries_ready, at_once, nullptr));
        opened->handle = nullptr;
    } else if (S_out && qi && oi && mapped_ints)
        ZKC(zk_lookup_prove_begin_mapped_ints(&p.handle, S0.gpu_data, qi, S_out->gpu_data, oi, mapped_ints, r->val, T0.gpu_data, m0.gpu_data, low, beta.val, u[0].val, vs[0].val,
                                              D, N, (int)k, nullptr));
    else if (S_out && oi && mapped_ints)
        ZKC(zk_lookup_prove_begin_mapped_out_ints(&p.handle, S0.gpu_data, S_out->gpu_data, oi, mapped_ints, r->val, T0.gpu_data, m0.gpu_data, low, beta.val, u[0].val, vs[0].val,
                                                  D, N, (int)k, nullptr));
    else if (S_out) ZKC(zk_lookup_prove_begin_mapped(&p.handle, S0.gpu_data, S_out->gpu_data, r->val, T0.gpu_data, m0.gpu_data, low, beta.val, u[0].val, vs[0].val, D, N, (int)k, nullptr));
    else if (hint == &S0 && qi)
        ZKC(zk_lookup_prove_begin_hinted_ints(&p.handle, S0.gpu_data, qi, T0.gpu_data, m0.gpu_data, low, beta.val, u[0].val, vs[0].val, D, N, (int)k, nullptr));
    else if (hint) ZKC(zk_lookup_prove_begin_hinted(&p.handle, S0.gpu_data, T0.gpu_data, m0.gpu_data, hint->gpu_data, low, beta.val, u[0].val, vs[0].val, D, N, (int)k, nullptr));
    else ZKC(zk_lookup_prove_begin(&p.handle, S0.gpu_data, T0.gpu_data, m0.gpu_data, beta.val, u[0].val, vs[0].val, D, N, (int)k, nullptr));
    return p;
}

Fr_t tLookup_sumcheck_end(LookupPending& pd) {
    const uint D = pd.D, N = pd.N;
    const vector<Fr_t>&u = pd.u, &v = pd.v;
    const uint n1 = ceilLog2(D / N);               // phase-1 rounds
    const uint k = (uint)u.size();
    if (k == 0) {
        const Fr_t claim = pd.alpha + pd.alpha * pd.alpha;
        zk_record(claim);
        return claim;
    }
    Fr_t bm;
    std::vector<Fr_t> sums((size_t)k * 11);
    void* h = pd.handle;
    pd.handle = nullptr;
    ZKC(zk_lookup_prove_end(h, bm.val, sums[0].val));
    pd.keep.clear();
    // Every product of the rounds has a factor that is known in Montgomery form (alpha, the eq factors, the challenge, N / D), so it
    // is one Montgomery product and leaves the other factor's standard form; the polynomials are their four coefficients.
    using zk::Fr;
    auto load = [](const Fr_t& x) { Fr r; memcpy(r.v, x.val, 32); return r; };
    auto store = [](const Fr& x) { Fr_t r; memcpy(r.val, x.v, 32); return r; };
    const Fr one = load(kOne), half_m = zk::to_mont(load(TWO_INV));
    const Fr inv_ratio_m = zk::to_mont(load(Fr_t{{N, 0, 0, 0, 0, 0, 0, 0}} / Fr_t{{D, 0, 0, 0, 0, 0, 0, 0}}));
    Fr alpha_m = zk::to_mont(load(pd.alpha));
    const Fr alpha_sq = zk::mont_mul(alpha_m, load(pd.alpha));
    Fr alpha_sq_m = zk::to_mont(alpha_sq);
    Fr claim = zk::add(load(pd.alpha), alpha_sq);
    Fr C = zk::sub(alpha_sq, load(bm));
    std::vector<Fr_t> coefs(4);
    for (uint r = 0; r < k; ++r) {
        Fr s[11];
        memcpy(s, &sums[(size_t)r * 11], sizeof(s));
        const bool phase2 = r >= n1;
        const Fr ub = load(u[k - 1 - r]), vr = load(phase2 ? v[k - 1 - (r - n1)] : v[n1 - 1 - r]);
        const Fr ub_m = zk::to_mont(ub), vr_m = zk::to_mont(vr);
        const Fr one_m = zk::big_one_mont<8>();
        // eq(ub) = e0 + e1 x; p = eq(ub) q + (s3 + s4 x) + the rest
        const Fr e0 = zk::sub(one_m, ub_m), e1 = zk::sub(zk::dbl(ub_m), one_m);
        Fr q[3], c[4];
        for (int i = 0; i < 3; ++i) q[i] = zk::mont_mul(alpha_m, s[i]);
        if (phase2) {
            const Fr coef_m = zk::mont_mul(inv_ratio_m, alpha_sq_m);
            for (int i = 0; i < 3; ++i) q[i] = zk::add(q[i], zk::mont_mul(coef_m, s[5 + i]));
        }
        c[0] = zk::add(zk::mont_mul(e0, q[0]), s[3]);
        c[1] = zk::add(zk::add(zk::mont_mul(e0, q[1]), zk::mont_mul(e1, q[0])), s[4]);
        c[2] = zk::add(zk::mont_mul(e0, q[2]), zk::mont_mul(e1, q[1]));
        c[3] = zk::mont_mul(e1, q[2]);
        if (phase2) for (int i = 0; i < 3; ++i) c[i] = zk::sub(c[i], zk::mont_mul(inv_ratio_m, s[8 + i]));
        else c[0] = zk::add(c[0], zk::mont_mul(half_m, C));
        for (int i = 0; i < 4; ++i) coefs[i] = store(c[i]);
        zk_record(coefs);
        const Fr at_one = zk::add(zk::add(c[0], c[1]), zk::add(c[2], c[3]));
        if (!zk::equal(claim, zk::add(c[0], at_one))) throw std::runtime_error(phase2 ? "tLookup_phase2: claim != p(0) + p(1)" : "tLookup_phase1: claim != p(0) + p(1)");
        claim = c[3];
        for (int i = 2; i >= 0; --i) claim = zk::add(zk::mont_mul(vr_m, claim), c[i]);
        const Fr uv = zk::mont_mul(ub_m, vr);
        const Fr e_m = zk::to_mont(zk::add(zk::sub(zk::dbl(uv), zk::add(ub, vr)), one));        // eq(ub, vr)
        alpha_m = zk::mont_mul(alpha_m, e_m);
        if (phase2) alpha_sq_m = zk::mont_mul(alpha_sq_m, e_m);
        else C = zk::mont_mul(half_m, C);
    }
    zk_record(store(claim));
    return store(claim);
}

Fr_t tLookup_sumcheck(const FrTensor& S0, const FrTensor& T0, const FrTensor& m0, const Fr_t& alpha0, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v) {
    LookupPending p = tLookup_sumcheck_begin(S0, T0, m0, alpha0, beta, u, v);
    return tLookup_sumcheck_end(p);
}

LookupPending tLookup::prove_begin(const FrTensor& S, const FrTensor& m, const Fr_t& alpha, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v) {
    if (m.size != table.size) throw std::runtime_error("m.size != table.size");
    return tLookup_sumcheck_begin(S, table, m, alpha, beta, u, v);
}

LookupPending tLookupRange::prove_begin(const FrTensor& S, const FrTensor& m, const Fr_t& alpha, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v) {
    if (m.size != table.size) throw std::runtime_error("m.size != table.size");
    return tLookup_sumcheck_begin(S, table, m, alpha, beta, u, v, &S, low);
}
// what a proof over N table entries and D queries has to be for its table to be inverted ahead (anything else goes through prove_begin, which says what is wrong)
static bool can_open(uint D, uint N, const vector<Fr_t>& u, const vector<Fr_t>& v) {
    return N >= 2 && N == (1u << ceilLog2(N)) && D == (1u << ceilLog2(D)) && D % N == 0 && u.size() == ceilLog2(D) && v.size() == ceilLog2(D);
}
LookupPending tLookupRange::count_and_prove_begin(const FrTensor& S, std::unique_ptr<FrTensor>& m, bool inside, const Fr_t& alpha, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v, bool at_once, bool more) {
    if (!can_open(S.size, table.size, u, v)) {
        m.reset(new FrTensor(inside ? prep_inside(S) : prep(S)));
        return prove_begin(S, *m, alpha, beta, u, v);
    }
    const void* h = S.kept_ints();
    const void* ints = h ? zk_fr_fold_prepared_ints(h) : nullptr;
    LookupOpened opened;
    ZKC(zk_lookup_open(&opened.handle, table.gpu_data, beta.val, table.size, nullptr));
    m.reset(new FrTensor(table.size));
    CountedQueries c;
    if (inside) ZKC(zk_lookup_multiplicities(m->gpu_data, nullptr, nullptr, ints, S.gpu_data, low, len, S.size, table.size, 1, nullptr));
    else ZKC(zk_lookup_multiplicities_begin(&c.check, m->gpu_data, nullptr, nullptr, ints, S.gpu_data, low, len, S.size, table.size, nullptr));
    // The rounds ahead of the table do not wait for the counting.  From 2^24 queries on the first of them holds the compute units for 0.7 ms, though: the counting by more than
    // LDS beside it, and behind that what the caller queues next, come to an end when it does, and then run beside rounds that are bound by memory like them.  Behind the
    // counting a rescaling of 2^24 elements by 2^16, 2^17, 2^18, 2^19 and 2^20 takes 1.62, 1.70, 1.73, 1.81 and 1.97 ms instead of 1.69, 1.78, 1.76, 1.97 and 2.04, but by 2^14 1.66 instead of 1.59;
    // 2^23 by 2^18 1.02 instead of 0.94, and a lookup of 2^24 in 2^16 entries, which has nothing more to queue, 1.35 instead of 1.32.  A layer's rescalings, which others run beside: no difference.
    const bool ahead = !(more && S.size >= (1u << 24) && table.size > (1u << 15));
    LookupPending p = sumcheck_begin(S, table, *m, alpha, beta, u, v, &S, low, nullptr, nullptr, nullptr, &opened, ahead, at_once);
    c.settle();
    return p;
}
Fr_t tLookupRange::prove(const FrTensor& S, const FrTensor& m, const Fr_t& alpha, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v, vector<Polynomial>& proof) {
    LookupPending p = prove_begin(S, m, alpha, beta, u, v);
    return tLookup_sumcheck_end(p);
}

LookupPending tLookupRangeMapping::prove_begin(const FrTensor& S_in, const FrTensor& S_out, const FrTensor& m, const Fr_t& r, const Fr_t& alpha, const Fr_t& beta,
                                               const vector<Fr_t>& u, const vector<Fr_t>& v) {
    return prove_begin_on(S_in, S_out, m, r, alpha, beta, u, v, nullptr);
}
std::unique_ptr<FrTensor> tLookupRangeMapping::combined(const Fr_t& r) const {
    std::unique_ptr<FrTensor> T(new FrTensor(table.size));
    ZKC(zk_fr_add_mul_s(T->gpu_data, table.gpu_data, mapped_vals.gpu_data, r.val, T->size, nullptr));
    return T;
}
tLookupRangeMapping::MappedPending tLookupRangeMapping::map_and_prove_begin(const FrTensor& S_in, const Fr_t& r, const Fr_t& alpha, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v) {
    MappedPending p;
    if (!can_open(1u << ceilLog2(S_in.size), table.size, u, v)) {
        auto ym = map_queued(S_in);
        p.y.reset(new FrTensor(std::move(ym.first)));
        p.m.reset(new FrTensor(std::move(ym.second)));
        p.look = prove_begin(S_in, *p.y, *p.m, r, alpha, beta, u, v);
        return p;
    }
    const bool positions = !(S_in.kept_ints() && mapped_vals.kept_ints());      // (asked before anything else is queued only where the queries have an int32 form)
    LookupOpened opened;
    opened.table = combined(r);
    ZKC(zk_lookup_open(&opened.handle, opened.table->gpu_data, beta.val, table.size, nullptr));
    CountedQueries c;
    count(c, S_in, positions, false);
    if (S_in.size != (1u << ceilLog2(S_in.size)) && !S_in.kept_ints()) {          // neither waits for what is asked next
        opened.queries = padded(opened.keep, S_in, table, false, nullptr);
        opened.m = padded_m(opened.keep, *c.m, S_in.size);
    }
    (void)mapped_vals.kept_ints();          // one wait for this and the range check
    c.settle();
    p.y.reset(new FrTensor(gather(S_in, c, nullptr)));
    p.m = std::move(c.m);
    p.look = prove_begin_on(S_in, *p.y, *p.m, r, alpha, beta, u, v, &opened);
    return p;
}
// Queries padded to a power of two with the first table entry, which are accounted for in m[0] (tlookup.cu:502-510).  Queries and outputs that
// keep int32 forms are padded in that form; where the job reads nothing else (zk_lookup_ints_suffice) the padded field elements are not written at all.
FrTensor* tLookupRangeMapping::padded(std::vector<std::unique_ptr<FrTensor>>& keep, const FrTensor& t, const FrTensor& fill_from, bool ints, const void* fill_ints) const {
    const uint D = t.size, Dp = 1u << ceilLog2(D);
    FrTensor* p = new FrTensor(Dp);
    keep.emplace_back(p);
    if (!(ints && zk_lookup_ints_suffice(Dp, table.size))) ZKC(zk_fr_pad_from(p->gpu_data, t.gpu_data, D, Dp, fill_from.gpu_data, nullptr));
    if (ints) ZKC(zk_i32_pad_from(p->ints_for_producer(), zk_fr_fold_prepared_ints(t.kept_ints()), D, Dp, fill_ints, low, nullptr));
    return p;
}
FrTensor* tLookupRangeMapping::padded_m(std::vector<std::unique_ptr<FrTensor>>& keep, const FrTensor& m, uint D) const {
    keep.emplace_back(new FrTensor(m.size));
    const Fr_t more{{(1u << ceilLog2(D)) - D, 0, 0, 0, 0, 0, 0, 0}};
    ZKC(zk_fr_copy_add_first(keep.back()->gpu_data, m.gpu_data, more.val, m.size, nullptr));
    return keep.back().get();
}
LookupPending tLookupRangeMapping::prove_begin_on(const FrTensor& S_in, const FrTensor& S_out, const FrTensor& m, const Fr_t& r, const Fr_t& alpha, const Fr_t& beta,
                                                  const vector<Fr_t>& u, const vector<Fr_t>& v, LookupOpened* opened) {
    const uint D = S_in.size;
    if (m.size != table.size) throw std::runtime_error("m.size != table.size");
    // (what is made for an opened job stays with it until the proof has begun: after an error its kernels may still read it, and it is waited for)
    std::vector<std::unique_ptr<FrTensor>> own_keep;
    std::vector<std::unique_ptr<FrTensor>>& keep = opened ? opened->keep : own_keep;
    const FrTensor *si = &S_in, *so = &S_out, *mm = &m;
    if (D != (1u << ceilLog2(D))) {
        const bool out_ints = S_out.kept_ints() && mapped_vals.kept_ints(), in_ints = out_ints && S_in.kept_ints();
        if (opened && opened->queries) { si = opened->queries; mm = opened->m; }
        else {
            si = padded(keep, S_in, table, in_ints, nullptr);          // the first table entry is low
            mm = padded_m(keep, m, D);
        }
        so = padded(keep, S_out, mapped_vals, out_ints, out_ints ? zk_fr_fold_prepared_ints(mapped_vals.kept_ints()) : nullptr);
    }
    const uint N = mm->size;
    if (N != (1u << ceilLog2(N)) || si->size % N != 0) throw std::runtime_error("N is not power of 2, or D is not divisible by N");
    // S_com = S_in + r * S_out (tlookup.cu:517) is formed by the job itself; T_com is small
    if (mapped_vals.size != table.size) throw std::runtime_error("Incompatible dimensions");
    std::unique_ptr<FrTensor> own = opened ? std::move(opened->table) : combined(r);
    const FrTensor& T_com = *own;
    keep.push_back(std::move(own));
    LookupPending p = sumcheck_begin(*si, T_com, *mm, alpha, beta, u, v, si, low, so, &r, mapped_vals.kept_ints(), opened, false, opened != nullptr);
    p.keep = std::move(keep);
    return p;
}

Fr_t tLookup::prove(const FrTensor& S, const FrTensor& m, const Fr_t& alpha, const Fr_t& beta, const vector<Fr_t>& u, const vector<Fr_t>& v, vector<Polynomial>& proof) {
    if (m.size != table.size) throw std::runtime_error("m.size != table.size");
    return tLookup_sumcheck(S, table, m, alpha, beta, u, v);
}

Fr_t tLookupRangeMapping::prove(const FrTensor& S_in, const FrTensor& S_out, const FrTensor& m, const Fr_t& r, const Fr_t& alpha, const Fr_t& beta,
                                const vector<Fr_t>& u, const vector<Fr_t>& v, vector<Polynomial>& proof) {
    LookupPending p = prove_begin(S_in, S_out, m, r, alpha, beta, u, v);
    return tLookup_sumcheck_end(p);
}
