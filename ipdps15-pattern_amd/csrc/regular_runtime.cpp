// Handle-level generalized reduction with an application's own functors and
// keyed reduction objects: RegularRuntime (kmeans/regular/regular_runtime.h:
// 79-105, regular_runtime.cu:31-291) for any map_fp / reduce_fp pair.  The
// input and its unit offsets are copied to the device once; each start
// sizes the wavefront tables and the final records, runs the application
// table's kernels (api/gpu/regular_table.hpp) and reads the final records
// back, sorted by key bytes.
//
// The reference's RegularRuntime splits units over the CPU threads and GPUs
// by a speed profile, feeds the GPU from mapped host memory and merges the
// device objects on the host (regular_runtime.cu:98-286; its merge_device is
// never called, regular_runtime.cu:285); with one GPU holding the input,
// one start is one device pass and the object comes back whole.
#include <algorithm>
#include <cstring>
#include <utility>
#include <vector>

#include "pat_common.hpp"

namespace {

constexpr int64_t kDefaultKeys = 4096;
constexpr int64_t kDefaultRecordBytes = 256;
// Wavefronts: a run of at least 256 units each (four rounds of the lanes, so
// that an LDS table's set-up and its records' way out stay small beside
// them), and no more than eight per CU, beyond which the fold's rows grow and
// the map gains nothing.  Each holds a table of the object's full capacity in
// case its LDS table overflows: their number is also held to kTableWords, or
// to one per kUnitsFew units where that takes more, and halved as long as the
// device has not that much memory.
constexpr int kMaxWaves = 2048;
constexpr int64_t kUnitsPerWave = 256;
constexpr int64_t kUnitsFew = 4096;
constexpr int kMaxWavesFew = 1024;
constexpr int64_t kTableWords = 1LL << 28;
constexpr int kStatusWords = 8;
constexpr int64_t kFirstWords = 65536;  // final records read back together with the status: 256 KiB, about 5 us

int64_t pow2_at_least(int64_t v)
{
    int64_t p = 1;
    while (p < v) p <<= 1;
    return p;
}

}  // namespace

struct pat_regular {
    void *input = nullptr;
    int64_t input_bytes = 0, num_units = 0, unit_bytes = 0;
    int64_t *offsets = nullptr;
    const pat_gr_table *table = nullptr;
    int map_idx = 0, reduce_idx = 0;
    void *param = nullptr;
    int64_t param_bytes = 0;
    int64_t max_keys = kDefaultKeys, max_record_bytes = kDefaultRecordBytes;
    int lds_keys = 0;
    uint32_t *tables = nullptr;  // wave tables, wave counts, final buckets, slots
    int64_t tables_words = 0;
    uint32_t *matrix = nullptr;  // all 0 between starts
    int64_t matrix_words = 0;
    bool matrix_clear = false;
    uint32_t *final = nullptr;  // status then the final records, read back together
    int64_t final_words = 0;
    uint32_t *host = nullptr;  // pinned: the status and the first kFirstWords of records
    hipStream_t stream = nullptr;
    // last start: the records, back to back, and their places in key order
    bool have_result = false;
    std::vector<uint32_t> records;
    struct Place {
        uint64_t prefix;  // the key's first eight bytes, big-endian, zero-padded
        uint32_t at;
    };
    std::vector<Place> out;
    int64_t merges = 0, reruns = 0;
    int waves = 0;

    void release()
    {
        if (stream) (void)hipStreamSynchronize(stream);
        for (void *p : {input, (void *)offsets, param, (void *)tables, (void *)matrix, (void *)final})
            if (p) (void)pat::dev_free(p);
        if (host) (void)hipHostFree(host);
        if (stream) (void)hipStreamDestroy(stream);
    }

    // Table geometry: buckets (a power of two, twice the keys) and pool words
    // (a header, key and value per record).
    int64_t buckets() const { return pow2_at_least(2 * max_keys); }
    int64_t pool_words() const { return max_keys * (1 + (max_record_bytes + 3) / 4 + 1); }

    // The final record at word 'at': header, key and value, each in whole words.
    static int64_t record_words(uint32_t hdr) { return 1 + (int64_t)((hdr >> 16) + 3) / 4 + ((hdr & 0xffffu) + 3) / 4; }
    int key_size(uint32_t at) const { return (int)(records[at] >> 16); }
    int value_size(uint32_t at) const { return (int)(records[at] & 0xffffu); }
    const unsigned char *key(uint32_t at) const { return (const unsigned char *)(records.data() + at + 1); }
    const unsigned char *value(uint32_t at) const
    {
        return (const unsigned char *)(records.data() + at + 1 + (key_size(at) + 3) / 4);
    }

    // Sorts 'out' by key bytes: a byte-wise radix sort of the prefixes, least
    // byte first (bytes all keys share are skipped: 5,003 four-byte keys take
    // two passes, some 20 us, where comparing took 0.25 ms), then runs of one
    // prefix by the rest.
    void sort_places()
    {
        std::vector<Place> other(out.size());
        for (int shift = 0; shift < 64; shift += 8) {
            size_t first[257] = {0};
            for (const Place &e : out) first[(e.prefix >> shift & 255) + 1]++;
            if (*std::max_element(first + 1, first + 257) == out.size()) continue;
            for (int i = 0; i < 256; i++) first[i + 1] += first[i];
            for (const Place &e : out) other[first[e.prefix >> shift & 255]++] = e;
            out.swap(other);
        }
        auto rest = [this](const Place &a, const Place &b) {
            const int ka = key_size(a.at), kb = key_size(b.at);
            const int c = memcmp(key(a.at), key(b.at), (size_t)std::min(ka, kb));
            if (c || ka != kb) return c ? c < 0 : ka < kb;
            // one key with values of two sizes: two records
            const int va = value_size(a.at), vb = value_size(b.at);
            const int d = memcmp(value(a.at), value(b.at), (size_t)std::min(va, vb));
            return d ? d < 0 : va < vb;
        };
        for (size_t i = 0, j; i < out.size(); i = j) {
            for (j = i + 1; j < out.size() && out[j].prefix == out[i].prefix;) j++;
            if (j > i + 1) std::sort(out.begin() + (int64_t)i, out.begin() + (int64_t)j, rest);
        }
    }

    int grow(uint32_t **p, int64_t *have, int64_t words)
    {
        if (words <= *have) return PAT_OK;
        if (*p) (void)pat::dev_free(*p);
        *p = nullptr;
        *have = 0;
        if (pat::dev_malloc(p, sizeof(uint32_t) * (size_t)words) != hipSuccess) {
            (void)hipGetLastError();
            *p = nullptr;
            pat::set_error("pat_regular_start: hipMalloc of %lld table bytes failed", (long long)(4 * words));
            return PAT_ERR_NOMEM;
        }
        *have = words;
        return PAT_OK;
    }

    int start()
    {
        PAT_REQUIRE(table, PAT_ERR_STATE, "pat_regular_start: no application table (pat_regular_set_table)");
        const int64_t nb = buckets(), pw = pool_words();
        PAT_REQUIRE(nb <= (1 << 24) && pw < (1LL << 31), PAT_ERR_INVALID, "pat_regular_start: object too large");
        // a wavefront's words: its table, its column of the matrix, its count
        const int64_t per_wave = 2 * nb + pw + 1;
        const int64_t few = std::min<int64_t>(kMaxWavesFew, std::max<int64_t>(1, (num_units + kUnitsFew - 1) / kUnitsFew));
        const int64_t fit = std::max(few, kTableWords / per_wave);
        waves = (int)std::min<int64_t>(std::min<int64_t>(kMaxWaves, fit),
                                       std::max<int64_t>(1, (num_units + kUnitsPerWave - 1) / kUnitsPerWave));
        PAT_TRY(grow(&final, &final_words, kStatusWords + pw));
        // where memory is short, fewer wavefronts do
        for (;; waves = (waves + 1) / 2) {
            if (nb * waves > matrix_words) matrix_clear = false;
            int rc = grow(&tables, &tables_words, (nb + pw) * waves + (waves + (waves & 1)) + 3 * nb);
            if (rc == PAT_OK) rc = grow(&matrix, &matrix_words, nb * waves);
            if (rc == PAT_OK) break;
            if (rc != PAT_ERR_NOMEM || waves == 1) return rc;
            for (auto [p, words] : {std::make_pair(&tables, &tables_words), std::make_pair(&matrix, &matrix_words)}) {
                if (*p) (void)pat::dev_free(*p);
                *p = nullptr;
                *words = 0;
            }
        }
        // LDS table: buckets a power of two covering lds_keys (or the
        // kernels' largest), pool words for that many records
        int lnb = table->max_lds_buckets, lpw = table->max_lds_pool_words;
        if (lds_keys > 0) {
            lnb = (int)std::min<int64_t>(lnb, pow2_at_least(lds_keys));
            lpw = (int)std::min<int64_t>(lpw, (int64_t)lds_keys * (2 + (max_record_bytes + 3) / 4));
        }
        pat_gr_object o;
        o.layout = 0;
        o.data = input;
        o.offsets = offsets;
        o.unit_bytes = unit_bytes;
        o.num_units = num_units;
        o.param = param;
        // the final buckets first: they are 8-byte words
        o.final_buckets = (unsigned long long *)tables;
        o.slots = (int32_t *)(tables + 2 * nb);
        o.wave_counts = (int32_t *)(tables + 3 * nb);
        o.wave_tables = tables + 3 * nb + (waves + (waves & 1));
        o.matrix = matrix;
        o.status = (int32_t *)final;
        o.final_pool = final + kStatusWords;
        o.waves = waves;
        o.table_buckets = (int32_t)nb;
        o.table_pool_words = (int32_t)pw;
        o.lds_buckets = lnb;
        o.lds_pool_words = lpw;
        if (!matrix_clear) PAT_HIP(hipMemsetAsync(matrix, 0, sizeof(uint32_t) * (size_t)matrix_words, stream));
        matrix_clear = false;  // until the run has ended well: its fold leaves the matrix clear
        PAT_HIP(hipMemsetAsync(o.status, 0, kStatusWords * sizeof(int32_t), stream));
        const int rc = table->map_reduce(map_idx, reduce_idx, &o, stream);
        PAT_REQUIRE(rc == PAT_OK, rc,
                    "pat_regular_start: the table's kernels for map %d / reduce %d failed (%d)%s", map_idx, reduce_idx,
                    rc, rc == PAT_ERR_INVALID ? "; a table built against another version of the library is refused" : "");
        const int64_t head = std::min(pw, kFirstWords);
        PAT_HIP(hipMemcpyAsync(host, final, sizeof(uint32_t) * (size_t)(kStatusWords + head), hipMemcpyDeviceToHost,
                               stream));
        PAT_HIP(hipStreamSynchronize(stream));
        matrix_clear = true;
        int32_t st[kStatusWords];
        memcpy(st, host, sizeof(st));
        PAT_REQUIRE(!(st[0] & 1), PAT_ERR_UNSUPPORTED,
                    "pat_regular_start: a wavefront met more keys than the object holds (%lld keys of %lld bytes; "
                    "pat_regular_set_capacity)", (long long)max_keys, (long long)max_record_bytes);
        PAT_REQUIRE(!(st[0] & 2), PAT_ERR_UNSUPPORTED,
                    "pat_regular_start: one unit's values do not fit an empty LDS table");
        PAT_REQUIRE(!(st[0] & 4), PAT_ERR_UNSUPPORTED,
                    "pat_regular_start: a map's insert was refused after another of its inserts was taken; it "
                    "cannot run again without inserting twice (a larger LDS table avoids the refusal)");
        PAT_REQUIRE(!(st[0] & 8), PAT_ERR_UNSUPPORTED,
                    "pat_regular_start: the final object is full (%lld keys of %lld bytes; pat_regular_set_capacity)",
                    (long long)max_keys, (long long)max_record_bytes);
        merges = st[1];
        reruns = st[2];
        const int64_t words = st[4];
        PAT_REQUIRE(words >= 0 && words <= pw && st[3] >= 0 && st[3] <= nb, PAT_ERR_INVALID,
                    "pat_regular_start: damaged final table");
        records.resize((size_t)words);
        memcpy(records.data(), host + kStatusWords, sizeof(uint32_t) * (size_t)std::min(words, head));
        if (words > head) {
            PAT_HIP(hipMemcpyAsync(records.data() + head, final + kStatusWords + head,
                                   sizeof(uint32_t) * (size_t)(words - head), hipMemcpyDeviceToHost, stream));
            PAT_HIP(hipStreamSynchronize(stream));
        }
        // the records' places, sorted by key bytes (a prefix of a key first)
        out.clear();
        out.reserve((size_t)st[3]);
        for (int64_t at = 0; at < words;) {
            const int64_t need = record_words(records[(size_t)at]);
            PAT_REQUIRE(at + need <= words, PAT_ERR_INVALID, "pat_regular_start: damaged final table record");
            uint64_t prefix = 0;
            const unsigned char *k = key((uint32_t)at);
            for (int i = 0; i < 8; i++) prefix = prefix << 8 | (i < key_size((uint32_t)at) ? k[i] : 0);
            out.push_back(Place{prefix, (uint32_t)at});
            at += need;
        }
        sort_places();
        have_result = true;
        return PAT_OK;
    }
};

extern "C" {

int pat_regular_create(const void *input, int64_t input_bytes, int64_t num_units, int64_t unit_bytes,
                       const int64_t *offsets, pat_regular **out)
{
    PAT_REQUIRE(out && input && input_bytes > 0 && num_units > 0 && unit_bytes > 0, PAT_ERR_INVALID,
                "pat_regular_create: bad arguments");
    PAT_REQUIRE(unit_bytes <= input_bytes, PAT_ERR_INVALID, "pat_regular_create: units larger than the input");
    if (offsets) {
        for (int64_t i = 0; i < num_units; i++)
            PAT_REQUIRE(offsets[i] >= 0 && offsets[i] <= input_bytes - unit_bytes, PAT_ERR_INVALID,
                        "pat_regular_create: unit %lld at %lld + %lld bytes lies outside the %lld-byte input",
                        (long long)i, (long long)offsets[i], (long long)unit_bytes, (long long)input_bytes);
    } else {
        PAT_REQUIRE(num_units <= input_bytes / unit_bytes, PAT_ERR_INVALID,
                    "pat_regular_create: %lld units of %lld bytes exceed the %lld-byte input", (long long)num_units,
                    (long long)unit_bytes, (long long)input_bytes);
    }
    auto *h = new pat_regular();
    h->input_bytes = input_bytes;
    h->num_units = num_units;
    h->unit_bytes = unit_bytes;
    int rc = PAT_OK;
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) {
        h->stream = nullptr;
        pat::set_error("pat_regular_create: stream creation failed");
        rc = PAT_ERR_HIP;
    }
    auto am = [&](void **p, size_t b) {
        if (rc == PAT_OK && pat::dev_malloc(p, b) != hipSuccess) {
            (void)hipGetLastError();
            *p = nullptr;
            pat::set_error("pat_regular_create: hipMalloc of %zu bytes failed", b);
            rc = PAT_ERR_NOMEM;
        }
    };
    am(&h->input, (size_t)input_bytes);
    if (rc == PAT_OK && hipHostMalloc((void **)&h->host, sizeof(uint32_t) * (size_t)(kStatusWords + kFirstWords),
                                      hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        h->host = nullptr;
        pat::set_error("pat_regular_create: pinned memory for the read-back failed");
        rc = PAT_ERR_NOMEM;
    }
    if (offsets) am((void **)&h->offsets, sizeof(int64_t) * (size_t)num_units);
    if (rc == PAT_OK &&
        (hipMemcpyAsync(h->input, input, (size_t)input_bytes, hipMemcpyHostToDevice, h->stream) != hipSuccess ||
         (offsets && hipMemcpyAsync(h->offsets, offsets, sizeof(int64_t) * (size_t)num_units, hipMemcpyHostToDevice,
                                    h->stream) != hipSuccess) ||
         hipStreamSynchronize(h->stream) != hipSuccess)) {
        pat::set_error("pat_regular_create: copying the input failed");
        rc = PAT_ERR_HIP;
    }
    if (rc != PAT_OK) {
        h->release();
        delete h;
        return rc;
    }
    *out = h;
    return PAT_OK;
}

int pat_regular_set_table(pat_regular *h, const pat_gr_table *table)
{
    PAT_REQUIRE(h, PAT_ERR_INVALID, "pat_regular_set_table: null handle");
    PAT_REQUIRE(table && table->map_count > 0 && table->reduce_count > 0 && table->map_reduce &&
                    table->max_lds_buckets > 0 && table->max_lds_pool_words > 0,
                PAT_ERR_INVALID, "pat_regular_set_table: bad table");
    h->table = table;
    h->map_idx = h->reduce_idx = 0;
    h->have_result = false;
    return PAT_OK;
}

int pat_regular_set_capacity(pat_regular *h, int64_t max_keys, int64_t max_record_bytes, int lds_keys)
{
    PAT_REQUIRE(h, PAT_ERR_INVALID, "pat_regular_set_capacity: null handle");
    PAT_REQUIRE(max_keys > 0 && max_keys <= (1 << 22) && max_record_bytes > 0 && max_record_bytes <= 65535 &&
                    lds_keys >= 0,
                PAT_ERR_INVALID, "pat_regular_set_capacity: out of range");
    h->max_keys = max_keys;
    h->max_record_bytes = max_record_bytes;
    h->lds_keys = lds_keys;
    return PAT_OK;
}

int pat_regular_set_map_idx(pat_regular *h, int idx)
{
    PAT_REQUIRE(h, PAT_ERR_INVALID, "pat_regular_set_map_idx: null handle");
    PAT_REQUIRE(!h->table || (idx >= 0 && idx < h->table->map_count), PAT_ERR_UNSUPPORTED,
                "pat_regular_set_map_idx: map index %d not in the table", idx);
    h->map_idx = idx;
    return PAT_OK;
}

int pat_regular_set_reduce_idx(pat_regular *h, int idx)
{
    PAT_REQUIRE(h, PAT_ERR_INVALID, "pat_regular_set_reduce_idx: null handle");
    PAT_REQUIRE(!h->table || (idx >= 0 && idx < h->table->reduce_count), PAT_ERR_UNSUPPORTED,
                "pat_regular_set_reduce_idx: reduce index %d not in the table", idx);
    h->reduce_idx = idx;
    return PAT_OK;
}

int pat_regular_set_param(pat_regular *h, const void *param, int64_t param_bytes)
{
    PAT_REQUIRE(h && param_bytes >= 0 && (param || param_bytes == 0), PAT_ERR_INVALID,
                "pat_regular_set_param: bad argument");
    if (param_bytes != h->param_bytes) {
        if (h->param) (void)pat::dev_free(h->param);
        h->param = nullptr;
        h->param_bytes = 0;
        if (param_bytes > 0) {
            if (pat::dev_malloc(&h->param, (size_t)param_bytes) != hipSuccess) {
                (void)hipGetLastError();
                h->param = nullptr;
                pat::set_error("pat_regular_set_param: hipMalloc of %lld bytes failed", (long long)param_bytes);
                return PAT_ERR_NOMEM;
            }
        }
        h->param_bytes = param_bytes;
    }
    if (param_bytes > 0) {
        PAT_HIP(hipMemcpyAsync(h->param, param, (size_t)param_bytes, hipMemcpyHostToDevice, h->stream));
        PAT_HIP(hipStreamSynchronize(h->stream));
    }
    h->have_result = false;
    return PAT_OK;
}

int pat_regular_start(pat_regular *h)
{
    PAT_REQUIRE(h, PAT_ERR_INVALID, "pat_regular_start: null handle");
    h->have_result = false;
    return h->start();
}

int pat_regular_get_output(pat_regular *h, int64_t *num_keys, int64_t *key_bytes, int64_t *val_bytes, void *keys,
                           uint32_t *key_index, uint32_t *key_size, void *vals, uint32_t *val_index,
                           uint32_t *val_size)
{
    PAT_REQUIRE(h && num_keys, PAT_ERR_INVALID, "pat_regular_get_output: null argument");
    PAT_REQUIRE(h->have_result, PAT_ERR_STATE, "pat_regular_get_output: no result (pat_regular_start)");
    int64_t ko = 0, vo = 0, i = 0;
    for (const auto &e : h->out) {
        const int ks = h->key_size(e.at), vs = h->value_size(e.at);
        if (keys) memcpy((char *)keys + ko, h->key(e.at), (size_t)ks);
        if (vals) memcpy((char *)vals + vo, h->value(e.at), (size_t)vs);
        if (key_index) key_index[i] = (uint32_t)ko;
        if (val_index) val_index[i] = (uint32_t)vo;
        if (key_size) key_size[i] = (uint32_t)ks;
        if (val_size) val_size[i] = (uint32_t)vs;
        ko += ks;
        vo += vs;
        i++;
    }
    *num_keys = i;
    if (key_bytes) *key_bytes = ko;
    if (val_bytes) *val_bytes = vo;
    return PAT_OK;
}

int pat_regular_stats(pat_regular *h, int64_t *merges, int64_t *reruns, int *waves)
{
    PAT_REQUIRE(h, PAT_ERR_INVALID, "pat_regular_stats: null handle");
    if (merges) *merges = h->merges;
    if (reruns) *reruns = h->reruns;
    if (waves) *waves = h->waves;
    return PAT_OK;
}

int pat_regular_destroy(pat_regular *h)
{
    if (!h) return PAT_OK;
    h->release();
    delete h;
    return PAT_OK;
}

}  // extern "C"
