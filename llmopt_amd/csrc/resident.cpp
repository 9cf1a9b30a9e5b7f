#include "resident.h"

#include <string.h>

#include <algorithm>

namespace llmopt {
namespace {

// One sequence, hidden 576, behind 2048 tokens: 1, 2, 4, 30 layers take 19, 31, 54, 357 us resident and 23 us a layer by
// launches: resident layers are the faster ones from the first on.  But they leave other bits than the records launched one by one, and
// plans of one to three layers are what checks make that compare the two; those keep the launches, at up to 25 us a step.
constexpr size_t kLeastLayers = 4;

bool is(const DispatchRecord &record, const char *name, size_t buffers, size_t parameter_bytes) {
  return record.name == name && record.buffers.size() == buffers && record.parameters.size() == parameter_bytes;
}
bool is_one_of(const DispatchRecord &record, const char *name, size_t buffers, size_t parameter_bytes) {
  return is(record, name, buffers, parameter_bytes) || is(record, (std::string(name) + "_m4").c_str(), buffers, parameter_bytes);
}

const uint16_t *halves(const DispatchRecord &record, size_t index) {
  return reinterpret_cast<const uint16_t *>(record.buffers[index].device);
}

// The records that may stand beside a run: they read the buffers in front of `outputs` and write the others, the first `bytes`
// of each.
struct Beside {
  const char *name;
  size_t buffers, parameter_bytes, outputs;
  size_t (*bytes)(const DispatchRecord &record, size_t index);
};
size_t whole(const DispatchRecord &record, size_t index) { return record.buffers[index].length; }
size_t product(const DispatchRecord &record, size_t first, size_t second, size_t bytes) {
  return (size_t)param_u32(record, first) * param_u32(record, second) * bytes;
}
size_t head_bytes(const DispatchRecord &record, size_t index) {
  return index == 0 ? product(record, 0, 8, 2) : index == 4 ? (size_t)param_u32(record, 0) * 4 : index == 5 ? product(record, 0, 4, 2) : whole(record, index);
}
size_t first_stage_bytes(const DispatchRecord &record, size_t index) {
  return index == 4 ? (size_t)param_u32(record, 0) * 256 * 8 : head_bytes(record, index);
}
const Beside kBeside[] = {
    {"llmopt_embedding_f16", 3, 12, 2,
     [](const DispatchRecord &r, size_t i) { return i == 0 ? (size_t)param_u32(r, 0) * 8 : i == 1 ? whole(r, i) : product(r, 0, 8, 2); }},
    {"llmopt_rms_norm_f16_simd", 3, 12, 2, [](const DispatchRecord &r, size_t i) { return i == 1 ? whole(r, i) : product(r, 0, 4, 2); }},
    {"llmopt_add_f16", 3, 136, 2, [](const DispatchRecord &r, size_t i) { return i == 2 ? (size_t)param_u32(r, 0) * 2 : whole(r, i); }},
    {"llmopt_w4a16_lm_head_argmax_f16", 5, 16, 4, head_bytes},
    {"llmopt_w4a16_lm_head_argmax_extra_f16", 6, 16, 4, head_bytes},
    {"llmopt_w4a16_lm_head_argmax_stage1_f16", 5, 16, 4, first_stage_bytes},
    {"llmopt_w4a16_lm_head_argmax_stage1_extra_f16", 6, 16, 4, first_stage_bytes},
    {"llmopt_w4a16_lm_head_reduce", 2, 4, 1,
     [](const DispatchRecord &r, size_t i) { return (size_t)param_u32(r, 0) * (i == 0 ? 256 * 8 : 4); }},
};

struct Stream {  // rows as the next layer takes them
  const uint8_t *rows = nullptr, *partials = nullptr;
  uint32_t partial_count = 0;
};

class Finder {
 public:
  explicit Finder(const std::vector<DispatchRecord> &records) : records_(records) {}

  // Layers from record `first` on; the records that the whole ones take, 0 if there are none.
  size_t from(size_t first) {
    run_ = {};
    run_.first = first;
    size_t at = first, kept_layers = 0, kept_records = 0;
    Stream stream;
    scratch_.clear();
    size_t kept_scratch = 0;
    while (const size_t taken = layer(at, &stream)) {
      at += taken;
      if (stream.partial_count == 0) {  // a whole stream behind it: the run may end here
        kept_layers = run_.layers.size();
        kept_records = at - first;
        kept_scratch = scratch_.size();
        run_.args.x_out = reinterpret_cast<uint16_t *>(const_cast<uint8_t *>(stream.rows));
        out_ = stream.rows;
      }
    }
    run_.layers.resize(kept_layers);
    scratch_.resize(kept_scratch);
    run_.count = kept_records;
    run_.args.layer_count = (uint32_t)kept_layers;
    return kept_layers >= kLeastLayers && fits() && may_run_again() ? kept_records : 0;
  }
  const ResidentRun &run() const { return run_; }

 private:
  const std::vector<DispatchRecord> &records_;
  ResidentRun run_;
  struct Range {
    const uint8_t *device;
    size_t length;
    bool marked;
    bool overlaps(const Range &other) const { return device < other.device + other.length && other.device < device + length; }
    bool holds(const Range &other) const { return device <= other.device && other.device + other.length <= device + length; }
  };
  std::vector<Range> scratch_;  // what the launches of the run write and the resident launch does not
  const uint8_t *out_ = nullptr;

  void writes(const DispatchRecord &record, size_t index) {
    const bool marked = index < record.retained.size() && record.retained[index]->scratch;
    scratch_.push_back({record.buffers[index].device, record.buffers[index].length, marked});
  }

  size_t layer(size_t at, Stream *stream) {
    if (at + 1 >= records_.size()) return 0;
    const DispatchRecord &qkv = records_[at], &attention = records_[at + 1];
    if (!is(qkv, "llmopt_rms_w4a16_qkv_rotary_pack_q8_f16_g64", 16, 44)) return 0;
    ResidentArgs &a = run_.args;
    const bool first = run_.layers.empty();
    const uint32_t m = param_u32(qkv, 0), h = param_u32(qkv, 4), qd = param_u32(qkv, 8), kvd = param_u32(qkv, 12);
    if (param_u32(qkv, 16) != kvd || qd % 64 != 0 || kvd % 64 != 0 || kvd == 0) return 0;
    const uint32_t partial_count = param_u32(qkv, 24);
    if (first) {
      if (partial_count != 0) return 0;
      a.m = m;
      a.h = h;
      a.q_heads = qd / 64;
      a.kv_heads = kvd / 64;
      a.per_kv = a.q_heads / a.kv_heads;
      a.attention_epsilon = param_f32(qkv, 20);
      a.token_elements = param_u32(qkv, 36);
      a.token_stride = param_u32(qkv, 40);
      a.x_in = halves(qkv, 0);
      a.cosine = halves(qkv, 10);
      a.sine = a.cosine + (size_t)m * 64;
      a.new_slots = reinterpret_cast<const uint32_t *>(qkv.buffers[14].device);
      a.pool = qkv.buffers[15].device;
      if (attention.buffers.size() < 9 || attention.parameters.size() < 68) return 0;
      a.slots = reinterpret_cast<const uint32_t *>(attention.buffers[4].device);
      a.past_lengths = reinterpret_cast<const uint32_t *>(attention.buffers[7].device);
      a.slot_offsets = reinterpret_cast<const uint32_t *>(attention.buffers[8].device);
      a.max_past = param_u32(attention, 64);
      a.scale = param_f32(attention, 48);
    } else if (qkv.buffers[0].device != stream->rows || partial_count != stream->partial_count ||
               (partial_count != 0 && qkv.buffers[1].device != stream->partials)) {
      return 0;
    }
    if (a.m != m || a.h != h || a.q_heads != qd / 64 || a.kv_heads != kvd / 64 || a.attention_epsilon != param_f32(qkv, 20) ||
        a.token_elements != param_u32(qkv, 36) || a.token_stride != param_u32(qkv, 40) || a.cosine != halves(qkv, 10) ||
        reinterpret_cast<const uint8_t *>(a.new_slots) != qkv.buffers[14].device || a.pool != qkv.buffers[15].device)
      return 0;
    ResidentLayer layer = {};
    for (int i = 0; i < 3; ++i) {
      layer.weight[i] = qkv.buffers[4 + 2 * i].device;
      layer.scale[i] = halves(qkv, 5 + 2 * i);
    }
    layer.attention_norm = halves(qkv, 3);
    layer.key_offset = param_u32(qkv, 28);
    layer.value_offset = param_u32(qkv, 32);

    const bool projecting = is(attention, "llmopt_attention_q8_paged_batched_w4a16_partial_g64", 11, 72);
    if (!projecting && !is(attention, "llmopt_attention_q8_paged_batched", 9, 68)) return 0;
    if (param_u32(attention, 0) != m || param_u32(attention, 4) != a.q_heads || param_u32(attention, 8) != a.kv_heads ||
        param_u32(attention, 16) != 64 || param_u32(attention, 20) != 0 || param_u32(attention, 28) != a.token_elements ||
        param_u32(attention, 32) != layer.key_offset || param_u32(attention, 36) != layer.value_offset ||
        param_u32(attention, 40) != 64 || param_u32(attention, 44) != a.token_stride || param_f32(attention, 48) != a.scale ||
        param_u32(attention, 52) > 1 || param_u32(attention, 60) != 0 || param_u32(attention, 64) != a.max_past)
      return 0;
    if (attention.buffers[0].device != qkv.buffers[11].device || attention.buffers[1].device != qkv.buffers[12].device ||
        attention.buffers[2].device != qkv.buffers[13].device || attention.buffers[3].device != a.pool ||
        attention.buffers[4].device != reinterpret_cast<const uint8_t *>(a.slots) ||
        attention.buffers[7].device != reinterpret_cast<const uint8_t *>(a.past_lengths) ||
        attention.buffers[8].device != reinterpret_cast<const uint8_t *>(a.slot_offsets))
      return 0;
    for (size_t b : {2, 11, 12, 13}) writes(qkv, b);
    writes(attention, 6);
    const size_t taken = projecting ? rest_in_sums(at, layer, stream) : rest_whole(at, layer, stream);
    if (taken != 0) run_.layers.push_back(layer);
    return taken;
  }

  // One SwiGLU width and epsilon in all layers.
  bool same_ffn(uint32_t mlp, float epsilon) {
    ResidentArgs &a = run_.args;
    if (run_.layers.empty()) {
      a.mlp = mlp;
      a.ffn_epsilon = epsilon;
    }
    return a.mlp == mlp && a.ffn_epsilon == epsilon;
  }

  size_t rest_in_sums(size_t at, ResidentLayer &layer, Stream *stream) {
    if (at + 2 >= records_.size()) return 0;
    const DispatchRecord &qkv = records_[at], &attention = records_[at + 1], &ffn = records_[at + 2];
    const ResidentArgs &a = run_.args;
    if (!is(ffn, "llmopt_sum_rms_w4a16_swiglu_down_partial_f16_g64", 11, 24) || param_u32(attention, 68) != a.h) return 0;
    const uint32_t mlp = param_u32(ffn, 4), slice = param_u32(ffn, 20);
    if (param_u32(ffn, 0) != a.m || param_u32(ffn, 8) != a.h || param_u32(ffn, 16) != a.q_heads || slice == 0 || mlp % slice != 0 ||
        !same_ffn(mlp, param_f32(ffn, 12)))
      return 0;
    if (ffn.buffers[0].device != qkv.buffers[2].device || ffn.buffers[1].device != attention.buffers[6].device) return 0;
    layer.weight[3] = attention.buffers[9].device;
    layer.scale[3] = halves(attention, 10);
    layer.ffn_norm = halves(ffn, 3);
    for (int i = 0; i < 3; ++i) {
      layer.weight[4 + i] = ffn.buffers[4 + 2 * i].device;
      layer.scale[4 + i] = halves(ffn, 5 + 2 * i);
    }
    writes(ffn, 2);
    writes(ffn, 10);
    *stream = {ffn.buffers[2].device, ffn.buffers[10].device, mlp / slice};
    return 3;
  }

  size_t rest_whole(size_t at, ResidentLayer &layer, Stream *stream) {
    if (at + 4 >= records_.size()) return 0;
    const DispatchRecord &qkv = records_[at], &attention = records_[at + 1], &out = records_[at + 2], &gate = records_[at + 3],
                         &down = records_[at + 4];
    const ResidentArgs &a = run_.args;
    if (!is_one_of(out, "llmopt_w4a16_linear_f16_g64", 5, 20) || !is(gate, "llmopt_rms_w4a16_dual_swiglu_f16_g64", 7, 16) ||
        !is_one_of(down, "llmopt_w4a16_down_add_f16_g64", 5, 16))
      return 0;
    if (param_u32(out, 0) != a.m || param_u32(out, 4) != a.h || param_u32(out, 8) != a.q_heads * 64 || param_u32(out, 12) != 1 ||
        param_u32(out, 16) != a.h || out.buffers[0].device != attention.buffers[6].device)
      return 0;
    // the stream, or the rows it is a copy of
    if (out.buffers[3].device != qkv.buffers[2].device &&
        !(param_u32(qkv, 24) == 0 && out.buffers[3].device == qkv.buffers[0].device))
      return 0;
    const uint32_t mlp = param_u32(gate, 4);
    if (param_u32(gate, 0) != a.m || param_u32(gate, 8) != a.h || !same_ffn(mlp, param_f32(gate, 12)) || param_u32(down, 0) != a.m ||
        param_u32(down, 4) != mlp || param_u32(down, 8) != a.h)
      return 0;
    if (gate.buffers[0].device != out.buffers[4].device || down.buffers[0].device != gate.buffers[6].device ||
        down.buffers[3].device != out.buffers[4].device)
      return 0;
    layer.weight[3] = out.buffers[1].device;
    layer.scale[3] = halves(out, 2);
    layer.ffn_norm = halves(gate, 1);
    for (int i = 0; i < 2; ++i) {
      layer.weight[4 + i] = gate.buffers[2 + 2 * i].device;
      layer.scale[4 + i] = halves(gate, 3 + 2 * i);
    }
    layer.weight[6] = down.buffers[1].device;
    layer.scale[6] = halves(down, 2);
    writes(out, 4);
    writes(gate, 6);
    writes(down, 4);
    *stream = {down.buffers[4].device, nullptr, 0};
    return 5;
  }

  bool fits() {
    const ResidentArgs &a = run_.args;
    if (!resident_ok(a.m, a.h, a.q_heads, a.kv_heads, a.mlp, a.layer_count)) return false;
    const auto bits = [](const void *pointer) { return reinterpret_cast<uintptr_t>(pointer); };
    // cache rows in 16-byte requests on 4-byte addresses, weights in 8-byte ones
    if ((bits(a.pool) & 3) != 0 || a.token_stride % 4 != 0 || a.token_elements % 64 != 0) return false;
    for (const ResidentLayer &layer : run_.layers)
      for (const uint8_t *weight : layer.weight)
        if ((bits(weight) & 7) != 0) return false;
    const Range result = result_rows();
    for (const Range &range : scratch_) {
      if (range.device == out_ && range.length >= result.length) continue;  // the run's result, which the resident launch writes too
      if (!range.marked || range.overlaps(result)) return false;
      for (size_t i = 0; i < records_.size(); ++i) {
        if (i >= run_.first && i < run_.first + run_.count) continue;
        for (const BoundBuffer &buffer : records_[i].buffers)
          if (range.overlaps({buffer.device, buffer.length, false})) return false;
      }
    }
    return true;
  }

  Range result_rows() const { return {out_, (size_t)run_.args.m * run_.args.h * 2, false}; }

  // A step whose resident launch gave up runs again from its first record, and the launch has left numbers where its result
  // belongs.  That comes to the same as a first run where no record writes what the step finds there and reads: the rows that
  // come in may be the result's only where a record in front writes all of them anew, and what is known of the records beside the
  // run must be enough to tell.  (The layers' own cache rows: each writes its new token's before it reads the sequence's.)
  bool may_run_again() const {
    std::vector<Range> read, written;  // (read: what the step finds there)
    const Range rows_in = {reinterpret_cast<const uint8_t *>(run_.args.x_in), result_rows().length, false};
    const Range pool = {run_.args.pool, records_[run_.first].buffers[15].length, false};
    const auto reads = [&](const Range &range) {
      for (const Range &earlier : written)
        if (earlier.holds(range)) return;
      read.push_back(range);
    };
    for (size_t i = 0; i < records_.size(); ++i) {
      const DispatchRecord &record = records_[i];
      if (i >= run_.first && i < run_.first + run_.count) {
        if (i == run_.first) reads(rows_in);
        for (const BoundBuffer &buffer : record.buffers) {
          const Range range = {buffer.device, buffer.length, false};
          const bool between = std::any_of(scratch_.begin(), scratch_.end(),
                                           [&](const Range &scratch) { return scratch.device != out_ && scratch.overlaps(range); });
          if (!between && buffer.device != rows_in.device && buffer.device != out_) reads(range);
        }
        if (i + 1 == run_.first + run_.count) written.push_back(result_rows());
        continue;
      }
      const auto known = std::find_if(std::begin(kBeside), std::end(kBeside), [&](const Beside &beside) {
        return is(record, beside.name, beside.buffers, beside.parameter_bytes);
      });
      if (known == std::end(kBeside)) return false;
      for (size_t b = 0; b < record.buffers.size(); ++b) {
        const Range range = {record.buffers[b].device, std::min(known->bytes(record, b), record.buffers[b].length), false};
        if (range.overlaps(pool)) return false;
        if (b < known->outputs) reads(range);
        else written.push_back(range);
      }
    }
    for (const Range &range : read)
      for (const Range &other : written)
        if (range.overlaps(other)) return false;
    return true;
  }
};

}  // namespace

bool find_resident_run(const std::vector<DispatchRecord> &records, ResidentRun *out) {
  Finder finder(records);
  for (size_t first = 0; first < records.size(); ++first)
    if (finder.from(first) != 0) {
      *out = finder.run();
      return true;
    }
  return false;
}

}  // namespace llmopt
