"""rf_design (include/rf_design.h): where the fields that ABI 9 and ABI 10 added
begin, its size, its ABI; test_emitted_forms.py checks them."""
ABI9, ABI10, SIZE, ABI = 260, 272, 288, 10
