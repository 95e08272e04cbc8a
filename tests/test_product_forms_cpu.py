"""Which products the generator marks row by row, and which it leaves to the
tuple walk: the rules of the `products` program, and its source whole."""
from srdatalog_hip import codegen, compiler, programs


def gens():
  prog = programs.PROGRAMS["products"]()
  arity = {d.name: d.arity for d in compiler.relation_decls(prog)}
  mir = compiler.compile_to_mir(prog)
  return {ep.rule: codegen.PipelineGen(ep, arity, i) for i, ep in enumerate(mir.pipelines())}


def test_every_rule_is_generated():
  prog = programs.PROGRAMS["products"]()
  src = codegen.generate_program_source("products", compiler.relation_decls(prog),
                                        compiler.compile_to_mir(prog))
  for rule in gens():
    assert f'{{"{rule}"' in src


def test_a_side_without_the_root_key_is_walked_by_tuples():
  g = gens()
  assert g["IndepPairs"].prod_kind() == 0 and g["IndepTriples"].prod_kind() == 0


def test_a_checked_root_key_is_walked_by_tuples():
  g = gens()
  assert g["RootNegation"].prod_kind() == 0 and g["RootFilter"].prod_kind() == 0


def test_a_union_adds_the_root_variable_once():
  """union_products knows one index column of the root variable."""
  g = gens()["RootTwice"]
  assert g.union_gen() is None and g.prod_kind() == 2
  assert g.gen_ext().strip() == '{"RootTwice", 2, nullptr, nullptr, 0, 0, 0, -1, 0}'


def test_unions_with_the_root_variable_in_the_head():
  """uni_minor, uni_row_col, uni_root_col of SrdPipelineExt."""
  g = gens()
  for rule, minor, row, root in (("KeyUnion", 0, 1, 0), ("KeyUnionMinor", 1, 0, 1)):
    assert g[rule].gen_ext().strip().endswith(f"_{rule}_union::k_desc, 1, {minor}, {row}, {root}, 0}}")
  assert g["Deep"].prod_kind() == 3 and g["Deep"].union_gen() is None
